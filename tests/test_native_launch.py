"""The extension module of the launch layer (csrc/torch_native.cpp): what it
takes gives bit for bit the results of the Python path, and what it does not
take still goes there, with the same errors."""

from __future__ import annotations

import sys

import pytest
import torch


class _Declines:
    """Stands in for the extension module and takes no call."""

    def __init__(self, real):
        self.decode_splits = real.decode_splits

    def __getattr__(self, name):
        return lambda *a: None


@pytest.fixture
def python_path(monkeypatch):
    from SSA import _lib

    def switch():
        stub = _Declines(_lib.native())
        monkeypatch.setattr(_lib, "native", lambda: stub)

    return switch


def test_declines_what_it_cannot_take():
    """CPU tensors, non-tensors and wrong argument counts return None; bind
    checks its arguments."""
    from SSA import _lib

    nat = _lib.native()
    x = torch.zeros(1, 2, 32, 64, dtype=torch.bfloat16)
    n = torch.tensor(1.5)
    assert nat.fwd(x, x, x, 0.1, n, n, True, 0, 0) is None
    assert nat.fwd(None, 3, "x", 0.1, n, n, True, 0, 0) is None
    assert nat.fwd() is None and nat.bwd(x) is None and nat.decode(1, 2) is None
    assert nat.varlen_fwd(x, x, x, n, 4, 0.1, n, n, True, 0, 0) is None
    with pytest.raises(TypeError):
        nat.bind(1, 2)
    with pytest.raises(ValueError):
        nat.bind(*[0] * 9)


def test_decode_splits():
    """256 workgroups, splits of at least 128 keys, short caches whole; the C
    ABI clamps and rounds the request as any other."""
    from SSA import _lib, ssa_decode_num_splits

    f = _lib.native().decode_splits
    assert f(1, 16, 16, 2048) == 16 and f(1, 4, 4, 8192) == 64 and f(1, 32, 8, 500) == 4
    assert f(16, 32, 8, 4096) == 2 and f(32, 32, 8, 8192) == 1 and f(1, 8, 8, 256) == 1
    assert f(1, 64, 1, 100000) == 128  # two groups of 32 heads
    assert f(0, 8, 8, 1000) == 1 and f(-1, 8, 8, 2**40) == 1
    assert ssa_decode_num_splits(1, 16, 16, 2048) == 16 and ssa_decode_num_splits(1, 16, 16, 2048, 3) == 3


def _views(t):
    yield "contiguous", t
    yield "s b h d", t.permute(2, 0, 1, 3).contiguous().permute(1, 2, 0, 3)
    wide = torch.zeros(*t.shape[:3], t.shape[3] + 8, dtype=t.dtype, device=t.device)
    wide[..., :t.shape[3]] = t
    yield "padded rows", wide[..., :t.shape[3]]
    odd = torch.zeros(*t.shape[:3], t.shape[3] + 4, dtype=t.dtype, device=t.device)
    odd[..., :t.shape[3]] = t
    yield "rows not 16-byte aligned", odd[..., :t.shape[3]]
    yield "transposed", t.transpose(2, 3).contiguous().transpose(2, 3)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 16), (torch.bfloat16, 32), (torch.float16, 64),
                                     (torch.bfloat16, 128), (torch.bfloat16, 256), (torch.float32, 16),
                                     (torch.float32, 64)])
@pytest.mark.parametrize("causal", [True, False])
def test_dense_matches_python_path(gpu, dtype, D, causal, python_path):
    from SSA import ssa_flash_attn_backward, ssa_flash_attn_forward

    B, Hq, Hkv, N = 2, 4, 2, 70
    g = torch.Generator(device=gpu).manual_seed(D)
    q, k, v, do = (torch.randn(B, h, N, D, generator=g, device=gpu).to(dtype) for h in (Hq, Hkv, Hkv, Hq))
    n, b = torch.tensor(1.5, device=gpu), torch.tensor([0.8], device=gpu)

    def both(ds):
        got = {}
        for name, qv in _views(q):
            kv = dict(_views(k))[name]
            print(f"[gpu case] native launch {dtype} D={D} {name} ds={ds}", file=sys.stderr, flush=True)
            out, m = ssa_flash_attn_forward(qv, kv, v, D ** -0.5, n, b, causal)
            grads = ssa_flash_attn_backward(qv, kv, v, out, dict(_views(do))[name], m, D ** -0.5, n, b, causal, ds)
            got[name] = (out, m, *grads)
        # scalars the fast path does not take: numbers, another dtype
        out, m = ssa_flash_attn_forward(q, k, v, D ** -0.5, 1.5, b.double(), causal)
        got["number scalars"] = (out, m)
        return got

    fast = [both(ds) for ds in (None, False)]
    python_path()
    slow = [both(ds) for ds in (None, False)]
    for f, s in zip(fast, slow):
        for name in f:
            for x, y in zip(f[name], s[name]):
                assert x.dtype == y.dtype and x.shape == y.shape and x.stride() == y.stride(), name
                assert torch.equal(x, y), name


@pytest.mark.gpu
def test_packed_and_decode_match_python_path(gpu, python_path):
    from SSA import ssa_decode_attention, ssa_flash_attn_varlen_backward, ssa_flash_attn_varlen_forward

    g = torch.Generator(device=gpu).manual_seed(3)
    T, Hq, Hkv, D = 150, 4, 2, 64
    q, k, v, do = (torch.randn(T, h, D, generator=g, device=gpu).bfloat16() for h in (Hq, Hkv, Hkv, Hq))
    cus = [torch.tensor([0, 70, 71, 150], dtype=dt, device=gpu) for dt in (torch.int32, torch.int64)]
    n, b = torch.tensor(1.5, device=gpu), torch.tensor(0.8, device=gpu)
    kc, vc = (torch.randn(3, Hkv, 100, D, generator=g, device=gpu).half() for _ in range(2))
    qd = torch.randn(3, Hq, 2 * D, generator=g, device=gpu).half()
    lens = [torch.tensor([100, 1, 37], dtype=dt, device=gpu) for dt in (torch.int32, torch.int64)]

    def all_calls():
        print("[gpu case] native launch packed / decode", file=sys.stderr, flush=True)
        got = []
        for cu in cus:
            out, m = ssa_flash_attn_varlen_forward(q, k, v, cu, 79, 0.125, n, b)
            got += [out, m, *ssa_flash_attn_varlen_backward(q, k, v, out, do, m, cu, 79, 0.125, n, b)]
        for ln in lens:
            for qv in (qd[..., :D], qd[..., ::2]):
                for splits in (0, 2):
                    got.append(ssa_decode_attention(qv, kc, vc, ln, 0.125, n, b, num_splits=splits))
        got += ssa_decode_attention(qd[..., :D], kc, vc, lens[0], 0.125, n, b, return_m=True)
        return got

    fast = all_calls()
    python_path()
    for x, y in zip(fast, all_calls()):
        assert x.shape == y.shape and x.dtype == y.dtype and torch.equal(x, y)


@pytest.mark.gpu
def test_errors_are_the_python_paths(gpu):
    from SSA import ssa_decode_attention, ssa_flash_attn_backward, ssa_flash_attn_forward

    q = torch.zeros(1, 3, 8, 64, dtype=torch.bfloat16, device=gpu)
    kv = torch.zeros(1, 2, 8, 64, dtype=torch.bfloat16, device=gpu)
    n = torch.tensor(1.5, device=gpu)
    with pytest.raises(AssertionError):
        ssa_flash_attn_forward(q, kv, kv, 0.1, n, n)  # 3 heads over 2
    with pytest.raises(AssertionError):
        ssa_flash_attn_forward(*[torch.zeros(1, 2, 8, 48, dtype=torch.bfloat16, device=gpu)] * 3, 0.1, n, n)
    with pytest.raises(ValueError):
        ssa_flash_attn_forward(q[:, :2], kv, kv.half(), 0.1, n, n)
    with pytest.raises(ValueError):
        ssa_flash_attn_forward(*[torch.zeros(1, 2, 8, 512, dtype=torch.bfloat16, device=gpu)] * 3, 0.1, n, n)
    out, m = ssa_flash_attn_forward(q[:, :2], kv, kv, 0.1, n, n)
    with pytest.raises(ValueError):
        ssa_flash_attn_backward(q[:, :2], kv, kv, out, out[:, :, :4], m, 0.1, n, n)
    with pytest.raises(ValueError):
        ssa_decode_attention(q[:, :2, 0], kv.float(), kv.float(), torch.ones(1, dtype=torch.int32, device=gpu), 0.1,
                             n, n)


@pytest.mark.gpu
def test_takes_the_plain_calls(gpu):
    """Every fast entry point runs a call in a plain layout itself, and leaves the
    odd ones (rows not 16-byte aligned, transposed, another dtype) to Python."""
    from SSA import _lib
    from SSA.ssa_hip_kernel import _current

    nat = _lib.native()
    g = torch.Generator(device=gpu).manual_seed(2)
    n = torch.tensor(1.5, device=gpu)
    views = dict(_views(torch.randn(1, 2, 40, 64, generator=g, device=gpu).bfloat16()))
    plain = {"contiguous", "s b h d", "padded rows"}
    for name, q in views.items():
        k = v = views["contiguous"]
        got = nat.fwd(q, k, v, 0.125, n, n, True, *_current())
        assert (got is not None) == (name in plain), name
        out, m = nat.fwd(k, k, v, 0.125, n, n, True, *_current())
        for ds_max in (0, -1, 1 << 30):
            grads = nat.bwd(k, k, v, out, q, m, 0.125, n, n, True, ds_max, *_current())
            assert (grads is not None) == (name in plain), (name, ds_max)
            assert grads is None or len(grads) == 5
    t = views["contiguous"][0].transpose(0, 1).contiguous()  # [T, H, D]
    cu = torch.tensor([0, 10, 40], dtype=torch.int32, device=gpu)
    out, m = nat.varlen_fwd(t, t, t, cu, 30, 0.125, n, n, True, *_current())
    assert len(nat.varlen_bwd(t, t, t, out, t, m, cu, 30, 0.125, n, n, True, 1 << 30, *_current())) == 5
    assert nat.varlen_fwd(t, t, t, cu.long(), 30, 0.125, n, n, True, *_current()) is None
    kc = views["contiguous"]
    qd, lens = kc[:, :, 0].contiguous(), torch.tensor([40], dtype=torch.int32, device=gpu)
    assert nat.decode(qd, kc, kc, lens, 0.125, n, n, 0, *_current())[0].shape == qd.shape
    assert nat.decode(qd.float(), kc, kc, lens, 0.125, n, n, 0, *_current()) is None


def _busy(x, ms):
    """About `ms` milliseconds of matrix products on the current stream."""
    for _ in range(ms):
        x = torch.mm(x, x)  # 8192^3: about a millisecond each in fp16
    return x


@pytest.mark.gpu
def test_runs_on_the_current_stream(gpu):
    """A launch on a side stream waits for that stream's work and for no other's."""
    from SSA import _lib, ssa_flash_attn_forward

    assert not isinstance(_lib.native(), _lib.PythonPath)
    g = torch.Generator(device=gpu).manual_seed(1)
    q, k, v, other = (torch.randn(1, 2, 64, 64, generator=g, device=gpu).bfloat16() for _ in range(4))
    load = torch.zeros(8192, 8192, device=gpu, dtype=torch.float16)
    n = torch.tensor(1.5, device=gpu)
    want, _ = ssa_flash_attn_forward(q, k, v, 0.125, n, n)
    _busy(load, 2)
    side = torch.cuda.Stream(device=gpu)
    late = other.clone()
    torch.cuda.synchronize()
    # the side stream's earlier work: one copy, long after the host has launched the forward
    with torch.cuda.stream(side):
        _busy(load, 30)
        late.copy_(q)
        got, _ = ssa_flash_attn_forward(late, k, v, 0.125, n, n)
    torch.cuda.synchronize()
    assert torch.equal(got, want)
    # no other stream's: the default stream is still busy when the side stream is done
    done, busy = torch.cuda.Event(), torch.cuda.Event()
    _busy(load, 60)
    busy.record()
    with torch.cuda.stream(side):
        got, _ = ssa_flash_attn_forward(q, k, v, 0.125, n, n)
        done.record()
    done.synchronize()
    assert not busy.query()
    torch.cuda.synchronize()
    assert torch.equal(got, want)
