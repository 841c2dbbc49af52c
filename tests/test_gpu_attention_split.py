"""The attention core over long contexts (scores by position tiles, softmax per row, weighted sum by dimension slices)
against the CPU oracle, bit for bit: whole models of one attention layer in four, so every logit and every cached row
downstream of an attention output would show a difference.

Sizes are where the kernels' paths change: contexts on both sides of the split's first position and of its 64-position
tiles, launches of 1, 4 and 8 rows and of whole and ragged prompt chunks, one to eight K/V heads with 1, 2, 3, 4 and 6
query heads each, head_dim 64, 128, 192 and 256, both forms of the weighted sum with more than one K/V head, a softmax
row of more than one 8192-value piece, and chunks in pieces of fewer rows (few score rows: states of long contexts)."""
import os
import sys

import numpy as np
import pytest

import oracle_lib as O

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qwen-3.8-in-rust_amd"))
import aqueduct as aq  # noqa: E402

pytestmark = pytest.mark.gpu
SEED = 411


@pytest.fixture(scope="module")
def ctx():
    return aq.Context(0)


def models(ctx, **kw):
    cfg = aq.tiny_config()
    for k, v in kw.items():
        setattr(cfg, k, v)
    tensors = aq.plan_tensors(aq.model_plan(cfg, aq.MIX_TINY, SEED))
    ocfg = O.AqModelConfig()
    for name, _ in O.AqModelConfig._fields_:
        setattr(ocfg, name, getattr(cfg, name))
    return cfg, aq.Model(ctx, cfg, tensors=tensors), O.Model(ocfg, tensors, threads=8)


@pytest.fixture(scope="module")
def tiny(ctx):
    return models(ctx, vocab=512)


@pytest.fixture(scope="module")
def wide(ctx):  # the 27B shape's head: 6 query heads of 256 on one K/V head
    return models(ctx, vocab=512, n_head=6, n_head_kv=1, head_dim=256, rope_dim=64)


def same(a, b):
    return np.array_equal(np.asarray(a, np.float32).view(np.uint32), np.asarray(b, np.float32).view(np.uint32))


def check(which, n, k, rounds, max_pos=None):
    cfg, gm, om = which
    ids = np.random.default_rng(n).integers(0, cfg.vocab, n).astype(np.uint32)
    g, o = aq.State(gm, k, max_pos or n + 200), O.State(om, k, n + 200)
    if k == 0:
        (ga, gl), (oa, ol) = g.prefill(ids, want_logits=True), o.prefill(ids, want_logits=True)
        assert ga == oa and same(gl, ol), "prompt logits"
        for i in range(rounds):
            (ga, gl), (oa, ol) = g.forward_token(ga, want_logits=True), o.forward_token(oa, want_logits=True)
            assert ga == oa and same(gl, ol), f"step {i}"
    else:
        x, y = g.spec_prefill(ids), o.spec_prefill(ids)
        assert x == y
        for i in range(rounds):
            assert g.drafts() == o.drafts(), f"round {i}"
            r = g.spec_round(x)
            assert r == o.spec_round(x), f"round {i}"
            x = r[1][-1]
    assert same(g.export(), o.export()), "state"


@pytest.mark.parametrize("n,k,rounds", [(250, 0, 12), (319, 0, 3), (250, 3, 6), (447, 7, 3), (701, 1, 2)])
def test_two_heads_of_64(tiny, n, k, rounds):
    print(f"split attention hd 64: prompt {n}, k {k}", flush=True)
    check(tiny, n, k, rounds)


@pytest.mark.parametrize("n,k,rounds", [(253, 0, 8), (384, 3, 4), (600, 7, 2)])
def test_six_heads_of_256(wide, n, k, rounds):
    print(f"split attention hd 256: prompt {n}, k {k}", flush=True)
    check(wide, n, k, rounds)


def test_softmax_rows_of_more_than_one_piece(tiny):
    print("split attention: 8,300 positions", flush=True)
    check(tiny, 8300, 3, 2)


@pytest.fixture(scope="module")
def heads(ctx):
    """Models by (n_head, n_head_kv, head_dim), one at a time."""
    made = {}

    def get(nh, nkv, hd):
        if (nh, nkv, hd) not in made:
            made.clear()
            made[nh, nkv, hd] = models(ctx, vocab=512, n_head=nh, n_head_kv=nkv, head_dim=hd, rope_dim=64)
        return made[nh, nkv, hd]

    return get


@pytest.mark.parametrize("nh,nkv,hd,n,k,rounds", [
    (12, 2, 256, 330, 3, 2),  # the wide weighted sum over two K/V heads, then 10 rows: wide scores, narrow sum
    (12, 2, 256, 371, 0, 3),  # its ragged last chunk (51 rows: 306 vectors)
    (8, 2, 128, 330, 3, 2), (8, 2, 128, 505, 0, 2),
    (4, 4, 128, 300, 3, 2),  # one query head per K/V head
    (12, 4, 192, 330, 3, 2), (12, 4, 192, 371, 7, 2),
    (8, 8, 192, 371, 0, 3),  # and the wide weighted sum with it
])
def test_head_shapes(heads, nh, nkv, hd, n, k, rounds):
    print(f"split attention {nh} heads on {nkv} of {hd}: prompt {n}, k {k}", flush=True)
    check(heads(nh, nkv, hd), n, k, rounds)


@pytest.mark.parametrize("which,max_pos,n,k", [("tiny", 400000, 400, 3), ("tiny", 1000000, 333, 0),
                                               ("wide", 400000, 400, 3), ("wide", 200000, 371, 0)])
def test_chunks_in_pieces(request, which, max_pos, n, k):
    """A state of so many positions that the score rows are for fewer than a chunk's 64 rows (192 MB of them: 31, 12, 20
    and 41 rows here): each chunk's attention runs in pieces, none of which divides it."""
    print(f"split attention in pieces, {which}: {max_pos} positions, prompt {n}, k {k}", flush=True)
    check(request.getfixturevalue(which), n, k, 2, max_pos)
