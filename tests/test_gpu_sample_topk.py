"""The selection of the first top_k candidates (sample.hip) against the oracle, where it can go wrong: vocabularies at the
edges of the 4096-key chunks, top_k at the ends of each form's range (1..128 by a bound, 129..512 by whole sorts), rows in
ascending and descending order and rows of few distinct values (the bound leaves more keys than are sorted, so the chunk
is sorted whole), infinities. Bar: the kept ids and probabilities and the dense row are the oracle's, bit for bit."""
import ctypes as C
import os
import sys

import numpy as np
import pytest

import oracle_lib as O

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qwen-3.8-in-rust_amd"))
import aqueduct as aq  # noqa: E402

pytestmark = pytest.mark.gpu


def rows_of(vocab):
    rng = np.random.default_rng(vocab)
    base = (rng.standard_normal(vocab) * 2.0).astype(np.float32)
    ties = rng.integers(0, 3, vocab).astype(np.float32)
    infs = base.copy()
    infs[rng.integers(0, vocab, max(1, vocab // 2))] = -np.inf
    infs[vocab - 1] = 1.5  # (a finite top: an all -inf row has no distribution)
    zeros = np.where(rng.integers(0, 2, vocab) == 1, np.float32(0.0), np.float32(-0.0)).astype(np.float32)
    return [base, np.sort(base), np.sort(base)[::-1].copy(), ties, infs, zeros]


@pytest.mark.parametrize("vocab", [1, 3, 255, 300, 4095, 4097, 20001, 70000])
@pytest.mark.parametrize("top_k", [1, 20, 128, 129, 512])
def test_first_candidates_equal_the_oracle(vocab, top_k):
    ctx = aq.Context(0)
    cfg = dict(temperature=0.9, top_k=top_k, seed=7)
    ds, os_ = aq.Sampler(ctx, aq.sampler_config(**cfg), vocab), O.Sampler(O.sampler_config(**cfg), vocab)
    lb, qb = aq.DeviceBuffer(ctx, vocab * 4), aq.DeviceBuffer(ctx, vocab * 4)
    qb.upload(np.full(vocab, 3.0, np.float32))
    for r, row in enumerate(rows_of(vocab)):
        print(f"case top-k vocab {vocab} top_k {top_k} row {r}", flush=True)
        lb.upload(row)
        ids, probs = ds.process(lb)
        oids, oprobs = os_.process(row)
        assert np.array_equal(ids, oids), f"row {r}: kept ids differ"
        assert np.array_equal(probs.view(np.uint32), np.asarray(oprobs, np.float32).view(np.uint32)), f"row {r}"
        ds.write_dense(qb)
        assert np.array_equal(qb.download(np.float32, vocab).view(np.uint32),
                              np.asarray(os_.write_dense(), np.float32).view(np.uint32)), f"row {r}: dense row"
        assert ds.draw() == os_.draw()
    for b in (lb, qb):
        b.free()
    ds.free()


def test_dense_row_after_queued_writes_to_its_buffer():
    """A row written while fills of the same buffer (and long ones before them) are still queued on the null stream, as a
    framework that clears its tensor leaves them, and on the context's stream: the row comes after them."""
    vocab, big = 70000, 256 << 20
    ctx = aq.Context(0)
    cfg = dict(temperature=0.9, top_k=40, seed=7)
    ds, os_ = aq.Sampler(ctx, aq.sampler_config(**cfg), vocab), O.Sampler(O.sampler_config(**cfg), vocab)
    lb, qb, long_ = aq.DeviceBuffer(ctx, vocab * 4), aq.DeviceBuffer(ctx, vocab * 4), aq.DeviceBuffer(ctx, big)
    row = rows_of(vocab)[0]
    lb.upload(row)
    ds.process(lb)
    os_.process(row)
    want = np.asarray(os_.write_dense(), np.float32)
    with open("/proc/self/maps") as f:  # the HIP runtime that the library runs on
        hip = C.CDLL(next(p for p in (line.split()[-1] for line in f) if "libamdhip64" in p))
    hip.hipMemsetAsync.argtypes = [C.c_void_p, C.c_int, C.c_size_t, C.c_void_p]
    for i in range(3):
        print(f"case dense row behind queued fills {i}", flush=True)
        for _ in range(100):
            assert hip.hipMemsetAsync(long_.p, i, big, None) == 0
        assert hip.hipMemsetAsync(qb.p, 0x41, vocab * 4, None) == 0
        ds.write_dense(qb)
        assert hip.hipStreamSynchronize(C.c_void_p(None)) == 0
        assert np.array_equal(qb.download(np.float32, vocab).view(np.uint32), want.view(np.uint32))
    for b in (lb, qb, long_):
        b.free()
    ds.free()
