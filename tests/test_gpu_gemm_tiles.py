"""The K-quant many-column kernels where their tiles and instances change, against the CPU oracle bit for bit: one to four
column tiles with a ragged last one, rows that end inside a 4-row weight tile or a 16-row tile, fewer super-blocks than
the LDS ring has stages, and row counts whose last pass over the CUs runs one column tile per work-group. And the
largest integers the matrix-core sums must hold exactly: random weight bytes and every code of one sign at its largest,
against activations of +-127 codes. And activation blocks too small for a finite scale."""
import os
import sys

import numpy as np
import pytest

import oracle_lib as O

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qwen-3.8-in-rust_amd"))
import aqueduct as aq  # noqa: E402

pytestmark = pytest.mark.gpu
KQ = [aq.Q4_K, aq.Q5_K, aq.Q6_K]
D_AT = {aq.Q4_K: (0, 2), aq.Q5_K: (0, 2), aq.Q6_K: (208,)}  # the block's f16 fields


@pytest.fixture(scope="module")
def ctx():
    return aq.Context(0)


def check(ctx, t, rows, cols, raw, x):
    n = x.shape[0]
    w = aq.Weight(ctx, t, rows, cols, raw)
    a = aq.Act(ctx, cols, n)
    a.set(x)
    a.quantize(t, n)
    got = aq.matmul(ctx, w, a, n)
    want = O.matmul(t, raw, rows, cols, x, threads=8)
    bad = int(np.sum(got.view(np.uint32) != np.asarray(want, np.float32).view(np.uint32)))
    assert bad == 0, f"{bad} of {got.size} outputs differ from the oracle"
    w.free()
    a.free()


def random_blocks(t, rows, cols, seed):
    """Random bytes, with finite f16 scales."""
    rng = np.random.default_rng(seed)
    raw = rng.integers(0, 256, (rows * cols // 256, aq.BLOCK[t][1]), dtype=np.uint8)
    for at in D_AT[t]:
        raw[:, at:at + 2] = rng.uniform(-1, 1, len(raw)).astype(np.float16).view(np.uint8).reshape(-1, 2)
    return raw.reshape(-1)


@pytest.mark.parametrize("t", KQ)
@pytest.mark.parametrize("rows,cols,n", [(1, 256, 64), (31, 1280, 17), (33, 512, 32), (50, 768, 48), (47, 1792, 49),
                                         (8200, 256, 64), (8230, 512, 41)])
def test_tiles_and_tails(ctx, t, rows, cols, n):
    print(f"gemm tiles type {t} {rows}x{cols} N={n}", flush=True)
    x = (np.random.default_rng(rows).standard_normal((n, cols)) * 2).astype(np.float32)
    check(ctx, t, rows, cols, random_blocks(t, rows, cols, 7 * rows + t), x)


@pytest.mark.parametrize("t", KQ)
@pytest.mark.parametrize("fill", [0xFF, 0x80, 0x7F, 0x00])
def test_largest_sums(ctx, t, fill):
    rows, cols, n = 20, 512, 24
    print(f"gemm largest sums type {t} fill {fill:#x}", flush=True)
    raw = random_blocks(t, rows, cols, fill).reshape(-1, aq.BLOCK[t][1])
    keep = [raw[:, at:at + 2].copy() for at in D_AT[t]]
    raw[: len(raw) // 2] = fill
    if t == aq.Q6_K:  # codes of 63 under scales of -128
        raw[len(raw) // 2 - 1, :192] = 0xFF
        raw[len(raw) // 2 - 1, 192:208] = 0x80
    for at, d in zip(D_AT[t], keep):
        raw[:, at:at + 2] = d
    x = np.ones((n, cols), np.float32)
    x[1::3] *= -3.0
    x[2::3, ::2] *= -1.0
    check(ctx, t, rows, cols, raw.reshape(-1), x)


@pytest.mark.parametrize("t", KQ)
@pytest.mark.parametrize("n", [9, 37, 64])
def test_tiny_activations(ctx, t, n):
    """Blocks whose largest magnitude is so small that -127 / max overflows (below about 3.7e-37: the reference's codes
    wrap to zero and d is zero), and on the other side of it, subnormal d: alone in a column, where the output shows
    them, and beside ordinary blocks."""
    rows, cols = 40, 1024
    print(f"gemm tiny activations type {t} N={n}", flush=True)
    rng = np.random.default_rng(n)
    x = rng.standard_normal((n, cols)).astype(np.float32)
    sizes = np.array([1e-42, 1e-39, 1e-38, 3e-37, 3.6e-37, 3.8e-37, 1e-36, 1e-34], np.float32)
    for c in range(n):  # each column: all blocks of one size, every other block, or one block
        for b in range(c % 3 // 2 * 2, 4 if c % 3 < 2 else 3, 1 + c % 3 % 2):
            blk = x[c, b * 256:(b + 1) * 256]
            x[c, b * 256:(b + 1) * 256] = blk / np.abs(blk).max() * sizes[c % len(sizes)]
    x[:, ::7] = 0.0  # (0 times an infinite scale)
    raw = random_blocks(t, rows, cols, 11 * n + t)
    assert np.isfinite(O.matmul(t, raw, rows, cols, x, threads=8)).all()
    check(ctx, t, rows, cols, raw, x)
