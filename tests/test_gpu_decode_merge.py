"""The decode step's two merge kernels (up to 4 splits, and more) against the
unsplit step: split counts around the border, around one lane per split (64)
and around whole rounds of the four waves, with empty splits and caches."""

from __future__ import annotations

import sys

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("splits", [2, 4, 5, 7, 8, 63, 64, 65, 80])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_splits_agree(gpu, D, splits, dtype):
    """out and m of a split step differ from the unsplit one's by fp32 rounding
    of the sums (m), and out by that and its rounding to 16 bits (half an ulp
    of either side: 2^-8 bf16, 2^-11 fp16 of the value)."""
    from SSA import ssa_decode_attention

    print(f"[gpu case] decode merge D={D} splits={splits} {dtype}", file=sys.stderr, flush=True)
    B, Hq, Hkv, cap = 3, 8, 2, 128 * splits
    g = torch.Generator(device=gpu).manual_seed(splits)
    q = torch.randn(B, Hq, D, generator=g, device=gpu).to(dtype)
    k, v = (torch.randn(B, Hkv, cap, D, generator=g, device=gpu).to(dtype) for _ in range(2))
    n, b = torch.tensor(4.0, device=gpu), torch.tensor(0.8, device=gpu)
    for lens in ([cap, cap // 2 + 1, 1], [0, cap - 1, 129]):
        ln = torch.tensor(lens, dtype=torch.int32, device=gpu)
        want, wm = ssa_decode_attention(q, k, v, ln, D ** -0.5, n, b, num_splits=1, return_m=True)
        got, gm = ssa_decode_attention(q, k, v, ln, D ** -0.5, n, b, num_splits=splits, return_m=True)
        torch.cuda.synchronize()
        fin = torch.isfinite(wm)
        assert torch.equal(fin, torch.isfinite(gm)) and torch.equal(gm[~fin], wm[~fin])
        assert ((gm - wm)[fin].abs() <= 1e-5 * (1 + wm[fin].abs())).all()
        ulp = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
        # P is rounded to 16 bits against each split's own maximum: 2 ulp of the largest |v| a row averages
        bound = 2 * ulp * want.float().abs() + 2 * ulp * v.float().abs().amax()
        assert ((got.float() - want.float()).abs() <= bound).all()
