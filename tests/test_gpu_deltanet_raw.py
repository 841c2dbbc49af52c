"""The isolated recurrence of a verify batch (deltanet_chunk.hip) against the oracle's steps: every head shape the library
takes, 1 to 8 rows, every count of kept rows (0: the state untouched), inputs at 4-byte and 16-byte alignment. Bar: the
outputs and the carried state equal bit for bit (the ordered sums and products are the oracle's). And outputs in the
memory of an input, equal to those in a buffer of their own."""
import ctypes as C
import os
import sys

import numpy as np
import pytest

import oracle_lib as O

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qwen-3.8-in-rust_amd"))
import aqueduct as aq  # noqa: E402

pytestmark = pytest.mark.gpu


class _At:
    """A device pointer `off` bytes into a buffer."""

    def __init__(self, buf, off):
        self.p = C.c_void_p(buf.p.value + off)


@pytest.mark.parametrize("dk,dv", [(8, 8), (16, 16), (32, 32), (64, 64), (128, 128), (128, 256), (64, 128)])
@pytest.mark.parametrize("t,keep", [(1, 0), (1, 1), (4, 2), (8, 0), (8, 1), (8, 7), (8, 8), (5, 5)])
def test_recurrence_equals_the_oracle(dk, dv, t, keep):
    nk, nv = 2, 4
    print(f"case recurrence {dk}x{dv} rows {t} kept {keep}", flush=True)
    ctx = aq.Context(0)
    L = O.lib()
    rng = np.random.default_rng(dk * 7 + dv + t + keep)
    s0 = (rng.standard_normal((nv, dk, dv)) * 0.3).astype(np.float32)
    q, k = [(rng.standard_normal((t, nk * dk)) / np.sqrt(dk)).astype(np.float32) for _ in range(2)]
    v = rng.standard_normal((t, nv * dv)).astype(np.float32)
    g = (-np.abs(rng.standard_normal((t, nv)))).astype(np.float32)
    beta = rng.random((t, nv), dtype=np.float32)
    so, want, s_keep = s0.copy(), np.zeros((t, nv * dv), np.float32), s0.copy()
    for i in range(t):
        for p in range(nv):
            kh = p % nk
            sp, o = np.ascontiguousarray(so[p]), np.zeros(dv, np.float32)
            L.or_deltanet_step(O.ptr(np.ascontiguousarray(q[i, kh * dk:(kh + 1) * dk])),
                               O.ptr(np.ascontiguousarray(k[i, kh * dk:(kh + 1) * dk])),
                               O.ptr(np.ascontiguousarray(v[i, p * dv:(p + 1) * dv])), float(g[i, p]), float(beta[i, p]),
                               O.ptr(sp), O.ptr(o), dk, dv)
            so[p], want[i, p * dv:(p + 1) * dv] = sp, o
        if i + 1 == keep:
            s_keep = so.copy()
    for off in (0, 4):
        bufs = []
        for arr in (q, k, v, g, beta, s0, np.zeros_like(want)):
            b = aq.DeviceBuffer(ctx, arr.nbytes + 16)
            b.upload(np.concatenate([np.zeros(off // 4, np.float32), arr.ravel()]))
            bufs.append(b)
        aq.deltanet_verify_commit_dev(ctx, nk, nv, dk, dv, t, keep, *[_At(b, off) for b in bufs])
        got = bufs[6].download(np.float32, want.size + off // 4)[off // 4:].reshape(want.shape)
        st = bufs[5].download(np.float32, s0.size + off // 4)[off // 4:].reshape(s0.shape)
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), f"outputs, offset {off}"
        assert np.array_equal(st.view(np.uint32), s_keep.view(np.uint32)), f"state, offset {off}"
        for b in bufs:
            b.free()


@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("t,keep", [(1, 1), (4, 0), (8, 3), (8, 8)])
@pytest.mark.parametrize("over", ["q", "k", "v", "v + 1 row", "q - 3"])
def test_output_over_an_input(d, t, keep, over):
    """The output in an input's own memory, whole or shifted: outputs and state as with a buffer of its own (nk = nv, so
    q, k, v and the output are the same size)."""
    n = 6
    print(f"case recurrence {d}x{d} rows {t} kept {keep}, output over {over}", flush=True)
    ctx = aq.Context(0)
    rng = np.random.default_rng(d + t + keep)
    s0 = (rng.standard_normal((n, d, d)) * 0.3).astype(np.float32)
    ins = {"q": rng.standard_normal((t, n * d)) / np.sqrt(d), "k": rng.standard_normal((t, n * d)) / np.sqrt(d),
           "v": rng.standard_normal((t, n * d)), "g": -np.abs(rng.standard_normal((t, n))), "b": rng.random((t, n))}
    off = {"v + 1 row": n * d, "q - 3": -3}.get(over, 0)
    got = []
    for alias in (False, True):
        bufs, ptrs = {}, {}
        for name, arr in list(ins.items()) + [("s", s0), ("o", np.zeros((t, n * d)))]:
            arr = np.asarray(arr, np.float32).ravel()
            bufs[name] = aq.DeviceBuffer(ctx, arr.nbytes + 8 * n * d)  # room on both sides for a shifted output
            bufs[name].upload(np.concatenate([np.zeros(n * d, np.float32), arr]))
            ptrs[name] = _At(bufs[name], 4 * n * d)
        at = over[0] if alias else "o"
        ptrs["o"] = _At(bufs[at], 4 * (n * d + (off if alias else 0)))
        aq.deltanet_verify_commit_dev(ctx, n, n, d, d, t, keep, *[ptrs[x] for x in "qkvgbso"])
        start = n * d + (off if alias else 0)
        out = bufs[at].download(np.float32, start + t * n * d)[start:]
        st = bufs["s"].download(np.float32, n * d + s0.size)[n * d:]
        got.append((out, st))
        for b in bufs.values():
            b.free()
    assert np.array_equal(got[0][0].view(np.uint32), got[1][0].view(np.uint32)), "outputs"
    assert np.array_equal(got[0][1].view(np.uint32), got[1][1].view(np.uint32)), "state"
