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
    ((16,), 256, 9, 0), ((8192,), 256, 17, 0),            # 512 and 1024 workgroups' worth
    ((8208,), 256, 16, 1), ((12,), 512, 33, 0),
    ((4096, 20, 4), 768, 48, 0), ((1024,), 1280, 500, 0),  # three waves; five
    ((1024,), 2048, 257, 0), ((520,), 2304, 320, 3),       # 8 waves; 9 superblocks in two rounds
    ((2052,), 3584, 70, 0), ((600,), 4352, 300, 0),        # two rounds of 7; three of 6, 6, 5
    ((7168,), 1024, 512, 0), ((64,), 1024, 512, 0),
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
