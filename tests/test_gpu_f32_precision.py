"""fp32 kernels against 64 bits: scores of long rows are summed in chains of 32
columns.

One fp32 chain of D products rounds D times, a tree of D / 32 chains of 32 about
32 + log2(D / 32) times, and rounding errors add up as their root: at head dim 256
a chain is off by 2.5 times as much.  The bounds lie 15 % above what the tree
measures and 15 % and more below one chain's; the seeds average over 8 heads x 4
draws."""

from __future__ import annotations

import sys

import pytest
import torch

from parity_util import oracle_fwd_bwd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,bounds", [(128, {"out": 1.25e-7, "dq": 2.85e-7, "dk": 3.6e-7}),
                                      (256, {"out": 1.36e-7, "dq": 3.1e-7, "dk": 3.85e-7})])
def test_score_sums(gpu, D, bounds):
    from SSA import ssa_flash_attn_backward, ssa_flash_attn_forward

    print(f"[gpu case] fp32 score sums D={D}", file=sys.stderr, flush=True)
    N, H, scale = 64, 8, D ** -0.5
    n, b = torch.tensor(1.5, device=gpu), torch.tensor(0.8, device=gpu)
    sums = {name: 0.0 for name in bounds}
    for seed in range(4):
        g = torch.Generator().manual_seed(seed)
        q, k, do, r = (torch.randn(1, H, N, D, generator=g) for _ in range(4))
        v, do = 0.9 * r + 0.4 * k, 0.9 * do + 0.4 * q
        q, k, v, do = (x.to(gpu) for x in (q, k, v, do))
        out, m = ssa_flash_attn_forward(q, k, v, scale, n, b)
        dq, dk, *_ = ssa_flash_attn_backward(q, k, v, out, do, m, scale, n, b)
        ref = oracle_fwd_bwd(q, k, v, do, scale, float(n), float(b), True)
        for name, got in (("out", out), ("dq", dq), ("dk", dk)):
            want = torch.from_numpy(ref[name])
            sums[name] += ((got.double().cpu() - want).norm() / want.norm()).item() ** 2 / 4
    for name, bound in bounds.items():
        assert sums[name] ** 0.5 <= bound, (name, sums[name] ** 0.5)
