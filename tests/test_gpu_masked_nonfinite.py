"""Masked pairs of the fp32-precision kernels (fp32; head dim 256) stay out of
every sum, whatever their operands hold.

A token's k, v, q or output gradient is made infinite or NaN; rows that the
causal mask (or the end of the sequence) keeps from it must come out bit for bit
as they do with finite values there.
"""

from __future__ import annotations

import math
import sys

import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [(torch.float32, 16), (torch.float32, 32), (torch.float32, 64), (torch.float32, 128), (torch.float32, 256),
          (torch.bfloat16, 256), (torch.float16, 256)]
BAD = [math.inf, -math.inf, math.nan]


def _run(q, k, v, do, causal):
    from SSA import ssa_flash_attn_backward, ssa_flash_attn_forward

    n, b = torch.tensor(1.5, device=q.device), torch.tensor(0.8, device=q.device)
    scale = q.shape[-1] ** -0.5
    out, m = ssa_flash_attn_forward(q, k, v, scale, n, b, causal)
    return (out, m, *ssa_flash_attn_backward(q, k, v, out, do, m, scale, n, b, causal))


def _inputs(gpu, dtype, D, N, seed):
    g = torch.Generator(device=gpu).manual_seed(seed)
    return [torch.randn(1, h, N, D, generator=g, device=gpu).to(dtype) for h in (4, 2, 2, 4)]


def _with(x, token, columns, value):
    y = x.clone()
    y[:, :, token, columns] = value
    return y


def _same(got, want):
    ulp = {torch.float32: 0.0, torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}[got.dtype]
    g, w = got.double(), want.double()
    return w.numel() == 0 or bool(((g - w).abs() <= ulp * w.abs() + 1e-5 * got.shape[-1] ** 0.5 * w.abs().max()).all())


@pytest.mark.parametrize("dtype,D", SHAPES)
@pytest.mark.parametrize("N,token", [(33, 17), (150, 64), (150, 149), (300, 131)])
@pytest.mark.parametrize("bad", BAD)
def test_causal_rows_before_and_after(gpu, dtype, D, N, token, bad):
    print(f"[gpu case] masked nonfinite {dtype} D={D} N={N} token={token} {bad}", file=sys.stderr, flush=True)
    q, k, v, do = _inputs(gpu, dtype, D, N, N + D)
    clean = _run(q, k, v, do, True)
    cols = [1, D - 1]
    # keys and values: queries before the token never see them
    for kk, vv in ((k, _with(v, token, cols, bad)), (_with(k, token, cols, bad), v)):
        got = _run(q, kk, vv, do, True)
        for i in (0, 2):  # out, dq
            assert _same(got[i][:, :, :token], clean[i][:, :, :token])
        assert _same(got[1][:, :, :token], clean[1][:, :, :token])
    got = _run(q, k, _with(v, token, cols, bad), do, True)
    assert not got[0][:, :, token:, cols].isfinite().any()
    rest = [c for c in range(D) if c not in cols]
    assert _same(got[0][..., rest], clean[0][..., rest])
    # queries and output gradients: keys after the token never meet them
    for qq, dd in ((q, _with(do, token, cols, bad)), (_with(q, token, cols, bad), do)):
        got = _run(qq, k, v, dd, True)
        for i in (3, 4):  # dk, dv
            assert _same(got[i][:, :, token + 1:], clean[i][:, :, token + 1:])
    # the output gradient weighs dv: the columns that it spoils, and no others
    got = _run(q, k, v, _with(do, token, cols, bad), True)
    assert not got[4][:, :, :token + 1, cols].isfinite().any()
    assert _same(got[4][..., rest], clean[4][..., rest])


@pytest.mark.parametrize("dtype,D", SHAPES)
@pytest.mark.parametrize("N", [33, 95])
def test_ragged_end(gpu, dtype, D, N):
    """Past the end of the sequence blocks repeat its last row at weight zero: an
    infinite last value row gives infinities, not NaN, and dK / dV of an
    infinite last output gradient likewise."""
    print(f"[gpu case] ragged nonfinite {dtype} D={D} N={N}", file=sys.stderr, flush=True)
    q, k, v, do = _inputs(gpu, dtype, D, N, N + D)
    clean = _run(q, k, v, do, False)
    got = _run(q, k, _with(v, N - 1, [3], math.inf), do, False)
    assert (got[0][..., 3] == math.inf).all()  # every weight is positive
    rest = [c for c in range(D) if c != 3]
    assert _same(got[0][..., rest], clean[0][..., rest])
    got = _run(q, k, v, _with(do, N - 1, [3], -math.inf), False)
    assert (got[4][..., 3] == -math.inf).all()
    assert _same(got[4][..., rest], clean[4][..., rest])
