"""The fp32-precision kernels (csrc/ssa_f32.hip) at the edges of their blocks.

A wave owns 32 rows and streams 32-row blocks, the waves of a workgroup share
stages of 1, 2 or 4 blocks (by head dim), dK/dV workgroups own 128 keys: the
lengths here sit on and beside those edges, against the fp64 oracle at the
bars of the other parity tests.
"""

from __future__ import annotations

import sys

import pytest
import torch

from parity_util import assert_parity, compare, make_inputs, oracle_fwd_bwd, scale_for

pytestmark = pytest.mark.gpu


def _grads(q, k, v, do, scale, causal):
    from SSA import ssa_flash_attn_backward, ssa_flash_attn_forward

    n = torch.tensor(1.5, device=q.device)
    b = torch.tensor(0.8, device=q.device)
    out, m = ssa_flash_attn_forward(q, k, v, scale, n, b, causal=causal)
    dq, dk, dv, dn, db = ssa_flash_attn_backward(q, k, v, out, do, m, scale, n, b, causal=causal)
    torch.cuda.synchronize()
    return {"out": out, "dq": dq, "dk": dk, "dv": dv, "dn": dn.item(), "db": db.item()}


@pytest.mark.parametrize("dtype,D", [(torch.float32, 16), (torch.float32, 32), (torch.float32, 64),
                                     (torch.float32, 128), (torch.float32, 256), (torch.bfloat16, 256),
                                     (torch.float16, 256)])
@pytest.mark.parametrize("N", [31, 33, 64, 65, 127, 161, 257])
@pytest.mark.parametrize("causal", [True, False])
def test_block_edges(gpu, dtype, D, N, causal):
    print(f"[gpu case] f32 mfma {dtype} D={D} N={N} causal={int(causal)}", file=sys.stderr, flush=True)
    q, k, v, do = make_inputs(1, 4, 2, N, D, dtype, gpu, "strided", seed=N * 7 + D)
    got = _grads(q, k, v, do, scale_for(D), causal)
    label = f"{dtype} D={D} N={N} causal={causal}"
    assert_parity(compare(got, oracle_fwd_bwd(q, k, v, do, scale_for(D), 1.5, 0.8, causal), scalars=()), label)
    ref = oracle_fwd_bwd(q, k, v, do, scale_for(D), 1.5, 0.8, causal, out_for_delta=got["out"])
    assert_parity(compare(got, ref), label + " [kernel-level]")


@pytest.mark.parametrize("causal", [True, False])
def test_fp16_weight_scale(gpu, causal):
    """fp16 at head dim 256 splits dS' in two fp16 halves under a running power
    of two per row: an output gradient that grows over six decades along the
    sequence moves it many times.  Every product and sum is then within about
    2^-22 of fp32, so dk and dq differ from the fp64 result by their own
    rounding to fp16 (2^-11 at most, normwise) and little more: each tensor as a
    whole here, and every dq row, of which the last outweigh the first by 10^6."""
    D, N = 256, 300
    print(f"[gpu case] fp16 weight scale causal={int(causal)}", file=sys.stderr, flush=True)
    q, k, v, do = make_inputs(1, 2, 2, N, D, torch.float16, gpu, "contig", seed=5)
    do = (do.float() * torch.logspace(-3, 3, N, device=gpu)[:, None]).to(torch.float16)
    got = _grads(q, k, v, do, scale_for(D), causal)
    ref = oracle_fwd_bwd(q, k, v, do, scale_for(D), 1.5, 0.8, causal, out_for_delta=got["out"])
    res = compare(got, ref, names=("dq", "dk"), scalars=())
    for name, st in res.items():
        assert st["finite"] and st["rel_rmse"] < 2.0 ** -11, (name, st)
    g, r = got["dq"].double().cpu(), torch.from_numpy(ref["dq"])
    rows = (g - r).norm(dim=-1) / (2.0 ** -11 * r.norm(dim=-1) + D ** 0.5 * 2.0 ** -25)
    # the first rows under the mask are differences that cancel in fp32
    assert rows[:, :, 8 if causal else 0:].max() < 1.1, rows.max()
