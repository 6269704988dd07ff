"""RMSNorm backward calls at the edges of the C interface: a gradient aligned to 8
bytes only, dx in place of x or dy, one partial and an odd dweight address."""

from __future__ import annotations

import ctypes
import sys

import pytest
import torch

pytestmark = pytest.mark.gpu


def _call(x, w, dy, rstd, dx, dw):
    from SSA import _lib

    rows, hidden = x.shape
    lib = _lib.lib()
    ws = torch.full((int(lib.ssa_rmsnorm_workspace_floats(rows, hidden)),), float("nan"), device=x.device)
    code = {torch.bfloat16: 0, torch.float16: 1, torch.float32: 2}[dy.dtype]
    a = _lib.RmsNormBwdArgs(x.data_ptr(), w.data_ptr(), dy.data_ptr(), rstd.data_ptr(), dx.data_ptr(), dw.data_ptr(),
                            ws.data_ptr(), rows, hidden, code)
    stream = torch.cuda.current_stream(x.device).cuda_stream
    assert lib.ssa_rmsnorm_bwd(ctypes.byref(a), ctypes.c_void_p(stream)) == 0
    torch.cuda.synchronize()
    return dx, dw


def _problem(gpu, rows, hidden, dtype=torch.float32):
    g = torch.Generator(device=gpu).manual_seed(rows + hidden)
    x, dy = (torch.randn(rows, hidden, generator=g, device=gpu) for _ in range(2))
    w = torch.randn(hidden, generator=g, device=gpu)
    return x, w, dy.to(dtype), torch.rsqrt(x.pow(2).mean(-1) + 1e-5)


@pytest.mark.parametrize("rows", [1, 64, 65, 200])
@pytest.mark.parametrize("hidden", [4, 260, 2048])
def test_calls(gpu, rows, hidden):
    print(f"[gpu case] RMSNorm backward calls {rows}x{hidden}", file=sys.stderr, flush=True)
    x, w, dy, rstd = _problem(gpu, rows, hidden)
    dx, dw = _call(x, w, dy, rstd, torch.empty_like(x), torch.empty_like(w))
    # dy at 8 bytes beyond a multiple of 16
    room = torch.zeros(dy.numel() + 4, device=gpu)
    for shift in (2, 4):
        view = room[shift:shift + dy.numel()].view_as(dy)
        view.copy_(dy)
        assert view.data_ptr() % 16 == (8 if shift == 2 else 0)
        for a, b in zip(_call(x, w, view, rstd, torch.empty_like(x), torch.empty_like(w)), (dx, dw)):
            assert torch.equal(a, b)
    # dx over x and over dy
    xi = x.clone()
    for a, b in zip(_call(xi, w, dy, rstd, xi, torch.empty_like(w)), (dx, dw)):
        assert torch.equal(a, b)
    di = dy.clone()
    for a, b in zip(_call(x, w, di, rstd, di, torch.empty_like(w)), (dx, dw)):
        assert torch.equal(a, b)
    # dweight at an address that takes no 16-byte store
    odd = torch.empty(hidden + 1, device=gpu)[1:]
    assert torch.equal(_call(x, w, dy, rstd, torch.empty_like(x), odd)[1], dw)
