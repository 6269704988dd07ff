"""The RMSNorm backward at the edges of its blocks: 4 rows per dx workgroup,
64 rows and 256 columns per weight-gradient partial, a column-group count that
changes above hidden sizes 1024 and 2048."""

from __future__ import annotations

import sys

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 5, 63, 64, 65, 1025])
@pytest.mark.parametrize("hidden", [4, 252, 260, 1024, 1028, 2048, 2052, 4096])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_backward_edges(gpu, rows, hidden, dtype):
    """dx and dw against fp64 on the same rounded dy.  fp32 sums of n terms in
    trees and short chains: at most 64 roundings deep, so 64 * 2^-24 = 4e-6 of
    the summed magnitudes bounds dw, and dx by the same with two factors."""
    from SSA.ssa_decoder import FusedRMSNormFn

    print(f"[gpu case] RMSNorm backward {rows}x{hidden} {dtype}", file=sys.stderr, flush=True)
    g = torch.Generator(device=gpu).manual_seed(rows * 4099 + hidden)
    x = torch.randn(rows, hidden, generator=g, device=gpu, requires_grad=True)
    w = (1 + 0.1 * torch.randn(hidden, generator=g, device=gpu)).requires_grad_(True)
    y = FusedRMSNormFn.apply(x, w, 1e-5, dtype)
    dy = torch.randn(rows, hidden, generator=g, device=gpu).to(dtype)
    dx, dw = torch.autograd.grad(y, (x, w), dy)
    x64, w64, dy64 = x.detach().double(), w.detach().double(), dy.double()
    r = torch.rsqrt(x64.pow(2).mean(-1, keepdim=True) + 1e-5)
    xh, gw = x64 * r, dy64 * w64
    ref_dx = r * (gw - xh * (gw * xh).mean(-1, keepdim=True))
    mag_dx = r * (gw.abs() + xh.abs() * (gw * xh).abs().mean(-1, keepdim=True))
    assert ((dx.double() - ref_dx).abs() <= 1e-5 * mag_dx).all()
    assert ((dw.double() - (dy64 * xh).sum(0)).abs() <= 4e-6 * (dy64 * xh).abs().sum(0)).all()
