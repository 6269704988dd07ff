"""fp16 at head dim 256: the weights of the outer products go in as two fp16
halves under a power of two, and each row keeps its own, so a row's gradient is
as exact beside rows of very different size as among its like.

Row by row against the fp64 oracle: rounding the result to fp16 moves a row by at
most 2^-11 of its norm (and 2^-25 an element below 2^-14); the halves add 2^-22.
Rows whose gradient overflows fp16 are only required not to disturb the others.
"""

from __future__ import annotations

import sys

import pytest
import torch

from parity_util import oracle_fwd_bwd

pytestmark = pytest.mark.gpu

D, SCALE, B_VAL = 256, 1 / 16, 0.8


def _check(gpu, q, k, v, do, n_val, names):
    from SSA import ssa_flash_attn_backward, ssa_flash_attn_forward

    q, k, v, do = (x.half().to(gpu)[None] for x in (q, k, v, do))
    n, b = torch.tensor(n_val, device=gpu), torch.tensor(B_VAL, device=gpu)
    out, m = ssa_flash_attn_forward(q, k, v, SCALE, n, b, False)
    got = dict(zip(("dq", "dk", "dv"), ssa_flash_attn_backward(q, k, v, out, do, m, SCALE, n, b, False)))
    ref = oracle_fwd_bwd(q, k, v, do, SCALE, n_val, B_VAL, False, out_for_delta=out)
    for name in names:
        g, r = got[name].double().cpu(), torch.from_numpy(ref[name])
        fits = r.abs().amax(-1) < 60000
        assert fits.sum() >= fits.numel() // 4
        err, size = (g - r).norm(dim=-1)[fits], r.norm(dim=-1)[fits]
        bound = (2.0 ** -11 + 2.0 ** -16) * size + D ** 0.5 * 2.0 ** -25
        worst = (err / bound).max().item()
        assert worst <= 1.0, (name, worst, (err / size.clamp_min(1e-30)).max().item())


def test_query_rows(gpu):
    """Output gradients of 2^13 and 2^-14 in turn, and values of 2^10: dQ rows 2^27
    apart in one 32-row block.  (Without the causal mask, whose first rows are
    differences that cancel in fp32.)"""
    print("[gpu case] d256 row scale dq", file=sys.stderr, flush=True)
    g = torch.Generator().manual_seed(1)
    N = 70
    q, k, v, do = (torch.randn(2, N, D, generator=g) for _ in range(4))
    size = torch.where(torch.arange(N) % 2 == 0, 2.0 ** 13, 2.0 ** -14)[:, None]
    _check(gpu, q, k, v * 2 ** 10, do.clamp(-3.5, 3.5) * size, 1.5, ["dq"])


@pytest.mark.parametrize("vsize,names", [(2.0 ** 10, ["dk"]), (1.0, ["dv"])])
def test_key_rows(gpu, vsize, names):
    """Keys that every query scores high and low in turn: probabilities 2^28 apart."""
    print(f"[gpu case] d256 row scale {names}", file=sys.stderr, flush=True)
    g = torch.Generator().manual_seed(2)
    N = 70
    u = torch.randn(D, generator=g)
    u = u / u.norm()
    q = 16 * u + 0.1 * torch.randn(2, N, D, generator=g)
    side = torch.where(torch.arange(N) % 2 == 0, 13.0, -13.0)[:, None]
    k = side * u + 0.1 * torch.randn(2, N, D, generator=g)
    v, do = (torch.randn(2, N, D, generator=g) for _ in range(2))
    _check(gpu, q, k, v * vsize, do.clamp(-3.5, 3.5) * 2 ** 13, 4.0, names)
