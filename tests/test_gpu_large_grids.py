"""Launches take fewer than 2^32 threads along x: grids of very many short
sequences fold over y, and the split decode's merge of very many heads takes its
narrow form."""

from __future__ import annotations

import sys

import pytest
import torch

pytestmark = pytest.mark.gpu


def test_fp32_backward_of_many_one_token_sequences(gpu):
    """2^23 (sequence, head) pairs of one token: 2^23 dK/dV workgroups of 512
    threads.  A lone token attends itself: out = v and dv = dout exactly."""
    from SSA import ssa_flash_attn_backward, ssa_flash_attn_forward

    B, H, D = 8192, 1024, 16
    print(f"[gpu case] fp32 backward, {B} x {H} sequences of one token", file=sys.stderr, flush=True)
    g = torch.Generator(device=gpu).manual_seed(0)
    q, k, v, do = (torch.randn(B, H, 1, D, generator=g, device=gpu) for _ in range(4))
    n, b = torch.tensor(1.5, device=gpu), torch.tensor(0.8, device=gpu)
    out, m = ssa_flash_attn_forward(q, k, v, 0.25, n, b)
    dq, dk, dv, dn, db = ssa_flash_attn_backward(q, k, v, out, do, m, 0.25, n, b)
    assert torch.allclose(out, v, rtol=1e-6, atol=0) and torch.allclose(dv, do, rtol=1e-6, atol=1e-6)
    assert dq.abs().max() < 1e-4 and dk.abs().max() < 1e-4  # dP - Delta: rounding only
    assert dn.isfinite() and db.isfinite()


def test_decode_merge_of_many_heads(gpu):
    """2^24 (sequence, head) pairs over five splits; the cache rows are shared by
    all sequences (stride 0)."""
    from SSA import ssa_decode_attention

    B, H, cap, D = 1 << 19, 32, 640, 32
    print(f"[gpu case] decode merge, {B} x {H} heads", file=sys.stderr, flush=True)
    g = torch.Generator(device=gpu).manual_seed(0)
    q = torch.randn(B, H, D, generator=g, device=gpu, dtype=torch.bfloat16)
    k, v = (torch.randn(1, 1, cap, D, generator=g, device=gpu).bfloat16().expand(B, 1, cap, D) for _ in range(2))
    lens = torch.full((B,), cap, dtype=torch.int32, device=gpu)
    n, b = torch.tensor(1.5, device=gpu), torch.tensor(0.8, device=gpu)
    got = ssa_decode_attention(q, k, v, lens, D ** -0.5, n, b, num_splits=5)
    pick = torch.tensor([0, 1, B // 2, B - 1], device=gpu)
    want = ssa_decode_attention(q[pick].contiguous(), k[:4], v[:4], lens[:4], D ** -0.5, n, b, num_splits=5)
    # the same partials merged in another order: fp32 sums, one rounding to bf16
    assert torch.allclose(got[pick].float(), want.float(), rtol=2.0 ** -7, atol=1e-6)
