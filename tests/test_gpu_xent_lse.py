"""The loss forward's log-sum-exp at the edges of its four-load step (4096
logits) and with infinities, NaN and the type's lowest value in a row."""

from __future__ import annotations

import ctypes
import sys

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V", [4, 1020, 1024, 3076, 4092, 4096, 4100, 8192, 20000])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_lse(gpu, V, dtype):
    from SSA import _lib

    print(f"[gpu case] cross-entropy lse V={V} {dtype}", file=sys.stderr, flush=True)
    inf, low = float("inf"), torch.finfo(dtype).min
    x = (torch.randn(12, V, generator=torch.Generator(device=gpu).manual_seed(V), device=gpu) * 5).to(dtype)
    x[1, V // 2] = -inf
    x[2] = -inf
    x[3] = low
    x[4, : V // 2] = -inf
    x[5] = torch.arange(V, device=gpu).to(dtype)  # a new maximum at nearly every logit
    x[6, 0] = -low
    x[7, -1] = inf
    x[8, 1] = float("nan")
    lab = torch.full((12,), -100, device=gpu)
    loss, lse = torch.empty(12, device=gpu), torch.empty(12, device=gpu)
    args = _lib.CrossEntropyArgs(x.data_ptr(), lab.data_ptr(), loss.data_ptr(), lse.data_ptr(), None, None, 12, V,
                                 0 if dtype == torch.bfloat16 else 1, 0)
    stream = torch.cuda.current_stream().cuda_stream
    _lib.check(_lib.lib().ssa_cross_entropy(ctypes.byref(args), ctypes.c_void_p(stream)), "ssa_cross_entropy")
    want = torch.logsumexp(x.double(), 1)
    # an infinite logit: exp(inf - inf), as the kernel has always answered
    assert lse[7:9].isnan().all() and lse[2] == -inf
    rest = torch.tensor([0, 1, 3, 4, 5, 6, 9, 10, 11], device=gpu)
    # every thread adds V / 256 terms and log2 of them meet: relative 2^-24 each, and the
    # exponentials' arguments carry 2^-24 of |x| <= 30 or of the distances that matter (< 90)
    tol = 2.0 ** -24 * (V / 256 + 12 + 2 * 90) + 2.0 ** -23 * want[rest].abs()
    assert ((lse[rest].double() - want[rest]).abs() <= tol).all()
