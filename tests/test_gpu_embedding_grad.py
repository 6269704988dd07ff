"""ssa_embedding_bwd against sums in 64 bits: table and column edges, one and
several lists (1024-token chunks, 2048 entries), frequent and neighbouring rows,
ids outside the table; and the calls that stay with PyTorch's own gradient."""

from __future__ import annotations

import ctypes
import sys

import pytest
import torch
import torch.nn.functional as F


def test_validation():
    from SSA import _lib

    lib, fake = _lib.lib(), 1 << 20
    for field, value, status in (("ids", None, 1), ("dy", None, 1), ("grad", None, 1), ("tokens", 0, 2),
                                 ("tokens", (1 << 26) + 1, 2), ("vocab", 0, 2), ("hidden", 6, 2), ("hidden", -4, 2),
                                 ("dy", fake + 8, 4), ("grad", fake + 4, 4), ("ids", fake + 4, 4)):
        a = _lib.EmbeddingBwdArgs(fake, fake, fake, 8, 64, 64)
        setattr(a, field, value)
        assert lib.ssa_embedding_bwd(ctypes.byref(a), None) == status, field
    assert lib.ssa_embedding_bwd(None, None) == 1


def test_plain_on_cpu_and_options():
    """CPU tensors and every option give nn.Embedding's own results."""
    from SSA.ssa_decoder import TokenEmbedding

    ids = torch.randint(50, (3, 40))
    for kw in ({}, {"padding_idx": 3}, {"scale_grad_by_freq": True}, {"sparse": True}, {"max_norm": 1.0}):
        torch.manual_seed(0)
        a = TokenEmbedding(50, 8, **kw)
        torch.manual_seed(0)
        b = torch.nn.Embedding(50, 8, **kw)
        ga, gb = (torch.autograd.grad(m(ids).square().sum(), m.weight)[0] for m in (a, b))
        assert torch.equal(a.weight, b.weight) and torch.equal(ga.to_dense(), gb.to_dense()), kw


@pytest.mark.gpu
@pytest.mark.parametrize("vocab,hidden", [(1, 4), (63, 260), (64, 256), (65, 252), (1000, 1028)])
@pytest.mark.parametrize("tokens", [1, 5, 1023, 1025, 2048, 2500, 5000])
@pytest.mark.parametrize("draw", ["even", "same", "halves", "outside"])
def test_sums(gpu, vocab, hidden, tokens, draw):
    from SSA.ssa_decoder import embedding_grad

    print(f"[gpu case] embedding grad {vocab}x{hidden} T={tokens} {draw}", file=sys.stderr, flush=True)
    g = torch.Generator(device=gpu).manual_seed(tokens)
    ids = torch.randint(vocab, (tokens,), generator=g, device=gpu)
    if draw == "same":
        ids.fill_(vocab // 2)
    elif draw == "halves":
        ids[: tokens // 2] = vocab - 1
    elif draw == "outside":
        ids[::3] = vocab + 5
        ids[1::7] = -1
    dy = torch.randn(tokens, hidden, generator=g, device=gpu)
    got = embedding_grad(dy, ids, vocab)
    ok = (ids >= 0) & (ids < vocab)
    want, mag, cnt = (torch.zeros(vocab, w, device=gpu, dtype=torch.float64) for w in (hidden, hidden, 1))
    want.index_add_(0, ids[ok], dy[ok].double())
    mag.index_add_(0, ids[ok], dy[ok].double().abs())
    cnt.index_add_(0, ids[ok], torch.ones_like(dy[ok][:, :1], dtype=torch.float64))
    # a sum of k terms in fp32, in any order: (k - 1) 2^-24 sum |x| at most
    assert ((got.double() - want).abs() <= 2.0 ** -24 * cnt * mag).all()
    assert torch.equal(got, embedding_grad(dy, ids, vocab))


@pytest.mark.gpu
@pytest.mark.parametrize("tokens", [99, 100, 3072, 3073])
def test_module(gpu, tokens):
    """Around the rule's ends, from a strided upstream gradient, int32 ids, a
    non-leaf weight, and a gradient of the gradient."""
    from SSA.ssa_decoder import TokenEmbedding

    print(f"[gpu case] token embedding T={tokens}", file=sys.stderr, flush=True)
    torch.manual_seed(tokens)
    m = TokenEmbedding(200, 64).to(gpu)
    ids = torch.randint(200, (tokens, 1), device=gpu)
    dy = torch.randn(64, 1, tokens, device=gpu).permute(2, 1, 0)
    for i in (ids, ids.to(torch.int32)):
        got, = torch.autograd.grad(m(i), m.weight, dy)
        want = torch.zeros(200, 64, device=gpu, dtype=torch.float64).index_add_(0, ids[:, 0], dy[:, 0].double())
        mag = torch.zeros(200, 64, device=gpu, dtype=torch.float64).index_add_(0, ids[:, 0], dy[:, 0].double().abs())
        assert ((got.double() - want).abs() <= 2.0 ** -24 * tokens * mag).all()
    assert torch.equal(m(ids), F.embedding(ids, m.weight))
    up = dy.clone().requires_grad_()
    first, = torch.autograd.grad(m(ids), m.weight, up, create_graph=True)
    second, = torch.autograd.grad(first.square().sum(), up)
    assert torch.allclose(second, 2 * F.embedding(ids, first.detach()))
