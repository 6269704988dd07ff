"""The forward's two workgroup sizes at head dim 128 (4 waves while every
128-row workgroup has a CU of its own, 8 beyond) compute each row the same way:
a few heads alone give bit for bit what they give inside a larger grid."""

from __future__ import annotations

import sys

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [97, 256, 321, 1025])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("dtype,n_val", [(torch.bfloat16, 1.5), (torch.float16, -3.484375)])
@pytest.mark.parametrize("layout", ["b h n d", "n b h d"])
def test_workgroup_sizes_agree(gpu, N, causal, dtype, n_val, layout):
    from SSA import ssa_flash_attn_forward

    print(f"[gpu case] forward waves N={N} causal={int(causal)} {dtype} {layout}", file=sys.stderr, flush=True)
    blocks = -(-N // 128)
    H = 256 // blocks + 8  # over 256 workgroups of 128 rows
    g = torch.Generator(device=gpu).manual_seed(N)
    shape = (1, H, N, 128) if layout == "b h n d" else (N, 1, H, 128)
    q, k, v = (torch.randn(shape, generator=g, device=gpu).to(dtype) for _ in range(3))
    if layout != "b h n d":
        q, k, v = (t.permute(1, 2, 0, 3) for t in (q, k, v))
    n, b = torch.tensor(n_val, device=gpu), torch.tensor(0.8, device=gpu)
    out, m = ssa_flash_attn_forward(q, k, v, 128 ** -0.5, n, b, causal)
    for h in (0, H - 4):
        s = slice(h, h + 4)
        out_s, m_s = ssa_flash_attn_forward(q[:, s], k[:, s], v[:, s], 128 ** -0.5, n, b, causal)
        assert torch.equal(out_s, out[:, s]) and torch.equal(m_s, m[:, s])
