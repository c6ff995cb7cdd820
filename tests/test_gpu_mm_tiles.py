"""The two kernels of products of more than 8 vectors, against the oracle bit for bit, at the edges of
the rule that picks between them (row groups x vector tiles above 512) and of their pipelines: one to
17 superblocks (a wave without one, whole rounds, a round with fewer waves, three rounds), one tile
per workgroup and many, ragged rows and vectors, several matrices, unaligned output rows, more than 64
vectors. The oracle is run on a sample of the rows of a large matrix."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

import oracle
from nibblemac_amd import pqtool
from nibblemac_amd.nmx import A8, NormIn
from tests.test_gpu_q4k import assert_bits_equal

pytestmark = pytest.mark.gpu


def chunk(dev, Ws, rows, cols, n, q, d, fs, pad):
    """nmx_q4k_matmul_chunk with output rows padded by `pad` floats."""
    vp, i = ctypes.c_void_p, ctypes.c_int
    fn = dev.lib.nmx_q4k_matmul_chunk
    fn.restype, fn.argtypes = i, [vp, i, vp, vp, vp, vp, i, i, vp, vp, vp]
    c = len(rows)
    Ys = [dev.zeros((n, r + pad), np.float32) for r in rows]
    dev.check(fn(dev.ctx, c, (vp * c)(*[w.ptr for w in Ws]), (i * c)(*rows),
                 (vp * c)(*[y.ptr for y in Ys]), (i * c)(*[r + pad for r in rows]), cols, n, q.ptr,
                 d.ptr, fs.ptr))
    dev.sync()
    out = [y.numpy() for y in Ys]
    for y in Ys:
        y.free()
    return out


CASES = [
    # rows of each matrix, cols, vectors, output row padding
    ((16,), 256, 9, 0), ((8192,), 256, 16, 0),             # one tile; 512, the last of q4k_mm_k
    ((8208,), 256, 16, 1), ((8192,), 256, 17, 0),          # 513 and 1024 of q4k_mmn_k
    ((12,), 512, 33, 0),
    ((4096, 20, 4), 768, 48, 0), ((1024,), 1280, 500, 0),  # three waves; five
    ((1024,), 2048, 257, 0), ((520,), 2304, 320, 3),       # 8 waves; 9 superblocks in two rounds
    ((2052,), 3584, 70, 0), ((600,), 4352, 300, 0),        # two rounds of 7; three of 6, 6, 5
    ((7168,), 1024, 512, 0), ((64,), 1024, 512, 0),
    ((2080,), 4096, 512, 0),  # 32 tiles per workgroup in two rounds: the most LDS
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "r%s_c%d_n%d_pad%d" % ("+".join(map(str, c[0])), *c[1:]))
def test_tiles_equal_oracle(dev, case):
    rows, cols, n, pad = case
    print(f"[case] mm tiles {case}", flush=True)
    rng = np.random.default_rng(cols + n)
    W = [pqtool.gauss_q4k(cols, k, r, cols, 0.02) for k, r in enumerate(rows)]
    q, d, fs = oracle.quant_a8(rng.standard_normal((n, cols)).astype(np.float32))
    dWs, (dq, dd, df) = [dev.to_device(w) for w in W], [dev.to_device(x) for x in (q, d, fs)]
    got = chunk(dev, dWs, rows, cols, n, dq, dd, df, pad)
    for w, r, y in zip(W, rows, got):
        tiles = np.unique(np.r_[0, 3, r // 4 - 1, rng.integers(0, r // 4, 12)])
        tiles = tiles[tiles < r // 4]
        some = np.ascontiguousarray(w.reshape(r // 4, -1)[tiles])
        want = oracle.q4k_matmul(some.ravel(), 4 * len(tiles), cols, q, d, fs, n)
        at = (4 * tiles[:, None] + np.arange(4)).ravel()
        assert_bits_equal(np.ascontiguousarray(y[:, at]), want, f"{r} x {cols}")
        assert not y[:, r:].any(), "padding columns written"
    for b in (*dWs, dq, dd, df):
        b.free()


def test_more_than_512_rows_refused(dev):
    """On the host, before anything is enqueued: the three matmul calls for chunks of rows."""
    print("[case] mm chunk refusals", flush=True)
    vp, i = ctypes.c_void_p, ctypes.c_int
    n, cols, rows = 513, 256, 32
    W, X = dev.zeros(rows // 4 * 576, np.uint8), dev.zeros((n, cols), np.float32)
    q, d, fs = dev.zeros((8, n, 32), np.int8), dev.zeros((8, n), np.float32), dev.zeros((8, n), np.float32)
    a8 = A8(q.ptr, d.ptr, fs.ptr)
    Y = [dev.zeros((n, rows), np.float32) for _ in range(2)]
    norm = NormIn(X.ptr, cols, None, 0, None, 0, X.ptr, 1e-6)
    one = ((vp * 1)(W.ptr), (i * 1)(rows), (vp * 1)(Y[0].ptr), (i * 1)(rows))
    mm, mmn, glu = (getattr(dev.lib, f"nmx_q4k_{x}_chunk") for x in ("matmul", "matmul_norm", "swiglu"))
    mmn.argtypes = [vp, i, vp, vp, vp, vp, i, i, ctypes.POINTER(NormIn), A8]
    glu.argtypes = [vp, vp, vp, i, i, i, vp, vp, vp, ctypes.POINTER(NormIn), vp, A8, A8, vp, vp]
    mm.argtypes = [vp, i, vp, vp, vp, vp, i, i, vp, vp, vp]
    assert mm(dev.ctx, 1, *one, cols, n, q.ptr, d.ptr, fs.ptr) == -1
    assert mmn(dev.ctx, 1, *one, cols, n, ctypes.byref(norm), a8) == -1
    assert glu(dev.ctx, W.ptr, W.ptr, rows, cols, n, q.ptr, d.ptr, fs.ptr, None, None, a8, a8, Y[0].ptr,
               Y[1].ptr) == -1
    dev.sync()
    assert not Y[0].numpy().any()
