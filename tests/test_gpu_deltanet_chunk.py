"""The DeltaNet mixer over prompt chunks (inputs, recurrence and output launches) against the CPU oracle, bit for bit:
whole models, so the logits, the recurrent states and the conv windows all show a difference. Chunks of 9 rows (the
fewest), 64, a ragged last one, and several in a row; every head shape a model can have; then a decode step and a verify round from
the state they leave."""
import os
import sys

import numpy as np
import pytest

import oracle_lib as O

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qwen-3.8-in-rust_amd"))
import aqueduct as aq  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    return aq.Context(0)


def same(a, b):
    return np.array_equal(np.asarray(a, np.float32).view(np.uint32), np.asarray(b, np.float32).view(np.uint32))


@pytest.mark.parametrize("dk,dv,nk,nv", [(64, 64, 2, 4), (128, 128, 1, 2), (64, 128, 1, 2), (128, 256, 1, 1)])
def test_prompt_chunks_equal_the_oracle(ctx, dk, dv, nk, nv):
    cfg = aq.tiny_config()
    cfg.vocab, cfg.dn_head_dim_k, cfg.dn_head_dim_v, cfg.dn_n_k_heads, cfg.dn_n_v_heads = 512, dk, dv, nk, nv
    tensors = aq.plan_tensors(aq.model_plan(cfg, aq.MIX_TINY, 97))
    ocfg = O.AqModelConfig()
    for name, _ in O.AqModelConfig._fields_:
        setattr(ocfg, name, getattr(cfg, name))
    gm, om = aq.Model(ctx, cfg, tensors=tensors), O.Model(ocfg, tensors, threads=8)
    for n in (9, 64, 75, 140):
        print(f"deltanet chunk {dk}x{dv} heads {nk}/{nv}: {n} tokens", flush=True)
        ids = np.random.default_rng(n).integers(0, cfg.vocab, n).astype(np.uint32)
        g, o = aq.State(gm, 3, n + 64), O.State(om, 3, n + 64)
        x = g.spec_prefill(ids)
        assert x == o.spec_prefill(ids)
        assert same(g.export(), o.export()), f"state after {n} tokens"
        assert g.spec_round(x) == o.spec_round(x)
        (ga, gl), (oa, ol) = g.forward_token(5, want_logits=True), o.forward_token(5, want_logits=True)
        assert ga == oa and same(gl, ol)
        assert same(g.export(), o.export()), f"state after a round and a step past {n} tokens"
