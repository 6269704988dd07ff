"""The backward reads the output gradient in its own strides: every layout of
the same values gives bit for bit the gradients of the contiguous tensor."""

from __future__ import annotations

import sys

import pytest
import torch

pytestmark = pytest.mark.gpu


def _layouts(x):
    """The values of x [B, H, N, D] in other layouts."""
    B, H, N, D = x.shape
    yield "s b h d", x.permute(2, 0, 1, 3).contiguous().permute(1, 2, 0, 3)
    yield "b n h d", x.transpose(1, 2).contiguous().transpose(1, 2)
    yield "last dim not 1", x.transpose(2, 3).contiguous().transpose(2, 3)
    wide = torch.zeros(B, H, N, 2 * D, dtype=x.dtype, device=x.device)
    wide[..., ::2] = x
    yield "every other element", wide[..., ::2]
    odd = torch.zeros(B * H * N * (D + 8) + 1, dtype=x.dtype, device=x.device)[1:].view(B, H, N, D + 8)
    odd[..., :D] = x
    yield "unaligned base", odd[..., :D]
    pad = torch.zeros(B, H, N, D + 4, dtype=x.dtype, device=x.device)
    pad[..., :D] = x
    yield "row stride not a multiple of 8", pad[..., :D]


@pytest.mark.parametrize("D,dtype", [(64, torch.bfloat16), (128, torch.float16), (64, torch.float32),
                                     (256, torch.bfloat16)])
def test_every_layout_gives_the_same_gradients(gpu, D, dtype):
    from SSA import ssa_flash_attention

    B, Hq, Hkv, N = 2, 4, 2, 77
    g = torch.Generator(device=gpu).manual_seed(D)
    q, k, v, do = (torch.randn(B, h, N, D, generator=g, device=gpu).to(dtype) for h in (Hq, Hkv, Hkv, Hq))
    n = torch.tensor(1.5, device=gpu, requires_grad=True)
    b = torch.tensor(0.8, device=gpu, requires_grad=True)
    leaves = [t.requires_grad_(True) for t in (q, k, v)] + [n, b]
    out = ssa_flash_attention(q, k, v, D ** -0.5, n, b)
    same = [do] + [do[:, :1].expand(B, Hq, N, D).contiguous()]
    want = [torch.autograd.grad(out, leaves, x, retain_graph=True) for x in same]
    views = [(name, x, want[0]) for name, x in _layouts(do)]
    views.append(("one head expanded", do[:, :1].expand(B, Hq, N, D), want[1]))
    for name, x, ref in views:
        print(f"[gpu case] dout layout {name} D={D} {dtype}", file=sys.stderr, flush=True)
        got = torch.autograd.grad(out, leaves, x, retain_graph=True)
        for a, r in zip(got, ref):
            assert torch.equal(a, r), name
