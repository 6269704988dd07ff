"""The dS' workspace of a backward: its size is weighed against the device's
headroom without Python objects, and where its allocation fails dq recomputes."""

from __future__ import annotations

import gc
import sys

import pytest
import torch

pytestmark = pytest.mark.gpu


class _Declines:
    def __init__(self, real):
        self.decode_splits, self.headroom = real.decode_splits, real.headroom

    def __getattr__(self, name):
        return lambda *a: None


@pytest.fixture(params=["extension", "python"])
def path(request, monkeypatch):
    """Both launch paths."""
    from SSA import _lib

    if request.param == "python":
        stub = _Declines(_lib.native())
        monkeypatch.setattr(_lib, "native", lambda: stub)
    return request.param


def _problem(gpu):
    """One whose workspace (270 MB) dwarfs its tensors (4 MB each)."""
    g = torch.Generator(device=gpu).manual_seed(0)
    q, k, v, do = (torch.randn(1, 16, 4096, 32, generator=g, device=gpu).bfloat16() for _ in range(4))
    n, b = torch.tensor(1.5, device=gpu), torch.tensor(0.8, device=gpu)
    return q, k, v, do, n, b


def _packed(gpu):
    """The same as a packed stream of one document."""
    q, k, v, do, n, b = _problem(gpu)
    q, k, v, do = (x[0].transpose(0, 1).contiguous() for x in (q, k, v, do))
    return q, k, v, do, n, b, torch.tensor([0, 4096], dtype=torch.int32, device=gpu)


def test_headroom(gpu):
    from SSA import _lib

    free, _ = torch.cuda.mem_get_info(gpu)
    want = free + torch.cuda.memory_reserved(gpu) - torch.cuda.memory_allocated(gpu)
    assert abs(_lib.native().headroom(0) - want) <= 64 << 20  # another process may come and go
    assert _lib.native().headroom(99) is None


def test_no_collections(gpu, path):
    """Weighing the workspace makes the interpreter collect nothing: 200 calls
    keep fewer objects alive than one young generation (700)."""
    from SSA import ssa_flash_attn_backward, ssa_flash_attn_forward

    print(f"[gpu case] ds headroom, collections, {path}", file=sys.stderr, flush=True)
    q, k, v, do, n, b = _problem(gpu)
    out, m = ssa_flash_attn_forward(q, k, v, 0.2, n, b)
    runs = []

    def seen(phase, info):
        if phase == "start":
            runs.append(info["generation"])

    gc.collect()
    gc.callbacks.append(seen)
    try:
        for _ in range(200):
            ssa_flash_attn_backward(q, k, v, out, do, m, 0.2, n, b)
    finally:
        gc.callbacks.remove(seen)
    torch.cuda.synchronize()
    assert len(runs) <= 1, runs


def test_failed_allocation_recomputes(gpu, path):
    """The allocator may not take the workspace: same gradients as without one; a
    workspace that is asked for still raises."""
    from SSA import (ssa_flash_attn_backward, ssa_flash_attn_forward, ssa_flash_attn_varlen_backward,
                     ssa_flash_attn_varlen_forward)

    print(f"[gpu case] ds headroom, failed allocation, {path}", file=sys.stderr, flush=True)
    q, k, v, do, n, b = _problem(gpu)
    out, m = ssa_flash_attn_forward(q, k, v, 0.2, n, b)
    want = ssa_flash_attn_backward(q, k, v, out, do, m, 0.2, n, b, ds=False)
    tq, tk, tv, td, n, b, cu = _packed(gpu)
    pout, pm = ssa_flash_attn_varlen_forward(tq, tk, tv, cu, 4096, 0.2, n, b)
    pwant = ssa_flash_attn_varlen_backward(tq, tk, tv, pout, td, pm, cu, 4096, 0.2, n, b, ds=False)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(gpu).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved(gpu) + (128 << 20)) / total, gpu)
    try:
        got = ssa_flash_attn_backward(q, k, v, out, do, m, 0.2, n, b)
        pgot = ssa_flash_attn_varlen_backward(tq, tk, tv, pout, td, pm, cu, 4096, 0.2, n, b)
        with pytest.raises(torch.OutOfMemoryError):
            ssa_flash_attn_backward(q, k, v, out, do, m, 0.2, n, b, ds=True)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0, gpu)
    for x, y in zip((*got, *pgot), (*want, *pwant)):
        assert torch.equal(x, y)
    # with room the workspace is taken: the other dQ kernel, whose sums differ in their last bits
    assert not torch.equal(ssa_flash_attn_backward(q, k, v, out, do, m, 0.2, n, b)[0], want[0])
