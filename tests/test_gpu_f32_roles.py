"""fp32 dK/dV on both sides of the rule that gives dK and dV workgroups of their
own (up to 128 workgroups of 128 keys, 256 under the causal mask): a key block's
dK and dV are the same sums in the same order either way, so a few heads alone
give bit for bit what they give inside a larger grid."""

from __future__ import annotations

import sys

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [16, 64, 128])
@pytest.mark.parametrize("causal,heads", [(True, 130), (False, 66)])
@pytest.mark.parametrize("N", [129, 256])
def test_roles_agree(gpu, D, causal, heads, N):
    from SSA import ssa_flash_attn_backward, ssa_flash_attn_forward

    print(f"[gpu case] fp32 roles D={D} causal={int(causal)} N={N}", file=sys.stderr, flush=True)
    g = torch.Generator(device=gpu).manual_seed(D + N)
    q, k, v, do = (torch.randn(1, heads, N, D, generator=g, device=gpu) for _ in range(4))
    n, b = torch.tensor(1.5, device=gpu), torch.tensor(0.8, device=gpu)

    def grads(s):
        out, m = ssa_flash_attn_forward(q[:, s], k[:, s], v[:, s], D ** -0.5, n, b, causal)
        return ssa_flash_attn_backward(q[:, s], k[:, s], v[:, s], out, do[:, s], m, D ** -0.5, n, b, causal)

    whole = grads(slice(None))  # 2 * heads workgroups of 128 keys: beyond the rule
    for h in (0, heads - 3):
        part = grads(slice(h, h + 3))
        for x, y in zip(part[:3], whole[:3]):
            assert torch.equal(x, y[:, h:h + 3])
    # dn and db: the sum over all heads from both routes, a few ulp of fp32 sums apart
    halves = [grads(slice(i, min(heads, i + 33))) for i in range(0, heads, 33)]
    for j in (3, 4):
        mag = sum(x[j].abs() for x in halves)
        assert (sum(x[j] for x in halves) - whole[j]).abs() <= 1e-5 * mag + 1e-6
