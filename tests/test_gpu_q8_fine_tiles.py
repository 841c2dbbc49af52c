"""The q8-fine matmul's block kernel (kq_q8f.hip) against the oracle at its edges: super-block counts around its stages of
four, rows around its tiles of 4, 8 and 32, columns around its fours and the 8-column pieces of a wider product, and one
column on both sides of the length where the block kernel takes it. Bar: equal bit for bit (every product and sum is the
oracle's, in its order)."""
import os
import sys

import numpy as np
import pytest

import oracle_lib as O

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qwen-3.8-in-rust_amd"))
import aqueduct as aq  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t", [aq.Q4_K, aq.Q5_K, aq.Q6_K])
@pytest.mark.parametrize("rows,nb", [(1, 1), (3, 3), (5, 4), (33, 5), (64, 8), (31, 9), (36, 24), (9, 25), (7, 30)])
def test_block_kernel_equals_the_oracle(t, rows, nb):
    ctx = aq.Context(0)
    cols = nb * 256
    spec = aq.synth_spec(t, rows, cols, seed=31 + t + rows, b=0.02)
    host = aq.synth_host(spec).view(np.uint8)
    w = aq.SynthWeight(ctx, spec)
    x = (np.random.default_rng(rows * 100 + nb).standard_normal((13, cols)) * 3.0).astype(np.float32)
    with aq.q8_fine(), O.q8_fine():
        for n in (1, 2, 3, 4, 5, 8, 13):
            print(f"case q8-fine block type {t} {rows}x{cols} columns {n}", flush=True)
            a = aq.Act(ctx, cols, n)
            a.set(x[:n])
            a.quantize(t, n)
            got = aq.matmul(ctx, w, a, n)
            want = O.matmul(t, host, rows, cols, x[:n], threads=4)
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), f"{n} columns"
            a.free()
    w.free()
