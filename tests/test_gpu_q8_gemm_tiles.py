"""The Q8_0 / Q4_0 many-column kernel at its edges against the CPU oracle, bit for bit: rows around its 32-row work-groups
and 16-row tiles, fewer 256-element steps than its ring has stages and just more, column tiles that are ragged or
missing, with random code bytes (Q8_0's -128 and every Q4_0 nibble among them) and scales of both signs from
the smallest f16 up, against ordinary and very small activations."""
import os
import sys

import numpy as np
import pytest

import oracle_lib as O

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qwen-3.8-in-rust_amd"))
import aqueduct as aq  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t", [aq.Q8_0, aq.Q4_0])
@pytest.mark.parametrize("rows,cols,n", [(1, 256, 9), (15, 512, 16), (17, 768, 17), (31, 1024, 33), (32, 1280, 48),
                                         (33, 2048, 64), (65, 512, 63), (300, 1792, 41), (48, 256, 10)])
@pytest.mark.parametrize("scale", [2.0, 1e-5])
def test_edges_equal_the_oracle(t, rows, cols, n, scale):
    print(f"case q8 gemm type {t} {rows}x{cols} N={n} scale {scale}", flush=True)
    ctx = aq.Context(0)
    rng = np.random.default_rng(rows * 131 + n)
    nblk = rows * cols // 32
    raw = rng.integers(0, 256, (nblk, aq.BLOCK[t][1]), dtype=np.uint8)
    d = (rng.uniform(-1, 1, nblk) * 2.0 ** rng.integers(-24, 4, nblk)).astype(np.float16)
    raw[:, :2] = d.view(np.uint8).reshape(-1, 2)
    raw = raw.reshape(-1)
    x = (rng.standard_normal((n, cols)) * scale).astype(np.float32)
    w, a = aq.Weight(ctx, t, rows, cols, raw), aq.Act(ctx, cols, n)
    a.set(x)
    a.quantize(t, n)
    got, want = aq.matmul(ctx, w, a, n), O.matmul(t, raw, rows, cols, x, threads=4)
    bad = int(np.sum(got.view(np.uint32) != np.asarray(want, np.float32).view(np.uint32)))
    assert bad == 0, f"{bad} of {got.size} outputs differ from the oracle"
    w.free()
    a.free()
