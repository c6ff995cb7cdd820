"""GPU parity of the prefill-chunk attention (more than 8 tokens: scores with a position per lane,
softmax in place, P.V with a dim per lane) against the step kernels over the same tokens in passes
of at most 8, which test_gpu_attn.py and the end-to-end tests pin.

Bar: bit-exact for the output, its A8 and both caches (every sum is the same ordered chain). Cases
at the tiles' edges: 9 rows, ragged row groups (3 heads per KV group), 64-position tiles entered and
left inside the chunk, softmax segments of 4096, caches past 8192 positions, head sizes 64 to 512."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

from nibblemac_amd.nmx import A8, AttnArgs
from tests.test_gpu_attn import cache_bytes
from tests.test_gpu_q4k import assert_bits_equal

pytestmark = pytest.mark.gpu


def fused_chunk(dev):
    fn = dev.lib.nmx_attn_fused_chunk
    fn.restype, fn.argtypes = ctypes.c_int, [ctypes.c_void_p, ctypes.POINTER(AttnArgs), ctypes.c_int]
    return fn


def passes(dev, host, shape, step, score_rows=0):
    """The chunk in passes of `step` tokens: o [n][nh hd], its A8 (codes, d, fsum per block and
    token), the caches. score_rows: through nmx_attn_fused_chunk with a workspace of so many rows."""
    n, nh, nkv, hd, max_ctx, kvt, pos0 = shape
    kc, vc = dev.to_device(host["kc"]), dev.to_device(host["vc"])
    const = {k: dev.to_device(host[k]) for k in ("q_norm", "k_norm", "cos", "sin")}
    nb, outs = nh * hd // 32, []
    for t0 in range(0, n, step):
        m = min(step, n - t0)
        q, k, v = (dev.to_device(host[x][t0:t0 + m]) for x in ("q", "k_in", "v_in"))
        pos = dev.to_device(np.array([pos0 + 3], np.int32))
        o = dev.zeros((m, nh * hd), np.float32)
        a8 = (dev.zeros((nb, m, 32), np.int8), dev.zeros((nb, m), np.float32),
              dev.zeros((nb, m), np.float32))
        sc = dev.zeros((score_rows or m, nh, max_ctx), np.float32)
        a = AttnArgs(m, nh, nkv, hd, hd // 4, max_ctx, q.ptr, k.ptr, v.ptr, const["q_norm"].ptr,
                     const["k_norm"].ptr, 1e-6, np.float32(1.0 / np.sqrt(hd)), const["cos"].ptr,
                     const["sin"].ptr, kc.ptr, vc.ptr, pos.ptr, t0 - 3, o.ptr,
                     A8(*[b.ptr for b in a8]), sc.ptr, kvt)
        if score_rows:
            dev.check(fused_chunk(dev)(dev.ctx, ctypes.byref(a), score_rows))
        else:
            dev.attn_prep(a)
            dev.attn(a)
        dev.sync()
        outs.append((o.numpy(), *[b.numpy() for b in a8]))
        for b in (q, k, v, pos, o, *a8, sc):
            b.free()
    return dict(o=np.concatenate([x[0] for x in outs]),
                **{k: np.concatenate([x[i] for x in outs], axis=1)
                   for i, k in ((1, "aq"), (2, "ad"), (3, "afs"))},
                kc=kc.numpy(), vc=vc.numpy())


CASES = [
    # n, query heads, KV heads, head size, max_ctx, kv dtype, position of token 0
    (9, 8, 2, 256, 1024, 0, 0),
    (64, 8, 2, 256, 1024, 0, 448),
    (64, 8, 2, 256, 1000, 0, 936),     # the last positions of a ragged cache
    (33, 8, 2, 256, 1024, 1, 40),
    (64, 8, 2, 256, 1024, 2, 63),
    (17, 6, 2, 128, 512, 0, 50),       # three heads per group: rows of a wave straddle tokens
    (12, 4, 4, 64, 256, 0, 10),
    (20, 8, 1, 512, 512, 1, 100),
    (40, 4, 2, 64, 8192, 0, 4080),     # rows across the first softmax segment's end
    (10, 2, 1, 64, 16384, 2, 9000),    # past the in-LDS step kernel, three segments
]


def make_host(rng, case):
    n, nh, nkv, hd, max_ctx, kvt, _ = case
    ang = rng.uniform(0, 2 * np.pi, (max_ctx, hd // 8))
    return dict(
        q=rng.standard_normal((n, nh, 2 * hd)).astype(np.float32),
        k_in=rng.standard_normal((n, nkv * hd)).astype(np.float32),
        v_in=rng.standard_normal((n, nkv * hd)).astype(np.float32),
        q_norm=rng.uniform(0.5, 1.5, hd).astype(np.float32),
        k_norm=rng.uniform(0.5, 1.5, hd).astype(np.float32),
        cos=np.cos(ang).astype(np.float32), sin=np.sin(ang).astype(np.float32),
        kc=cache_bytes(rng, kvt, nkv, max_ctx, hd), vc=cache_bytes(rng, kvt, nkv, max_ctx, hd),
    )


@pytest.mark.parametrize("case", CASES, ids=lambda c: "n%d_h%d_%d_hd%d_ctx%d_kv%d_pos%d" % c)
def test_chunk_equals_steps(dev, case):
    n, nh, nkv, hd, max_ctx, kvt, pos0 = case
    print(f"[case] attn chunk {case}", flush=True)
    host = make_host(np.random.default_rng(n + 7 * hd + pos0), case)
    want = passes(dev, host, case, 8)
    got = passes(dev, host, case, 64)
    for k in want:
        assert_bits_equal(got[k], want[k], k)


@pytest.mark.parametrize("case,score_rows", [
    ((130, 8, 2, 256, 512, 0, 20), 64),   # two whole slices and one of two rows
    ((512, 4, 2, 64, 640, 1, 100), 200),  # the most rows, a ragged last slice
    ((9, 6, 2, 128, 256, 2, 50), 4),      # fewer workspace rows than a pass of steps
], ids=lambda c: str(c).replace(" ", ""))
def test_slices_equal_steps(dev, case, score_rows):
    """nmx_attn_fused_chunk in slices of the scores workspace's rows."""
    print(f"[case] attn chunk slices {case} {score_rows}", flush=True)
    host = make_host(np.random.default_rng(sum(case)), case)
    want = passes(dev, host, case, 8)
    got = passes(dev, host, case, 512, score_rows)
    for k in want:
        assert_bits_equal(got[k], want[k], k)


def test_fused_chunk_refusals(dev):
    """On the host: a workspace of no rows or none at all, and more rows than NMX_CHUNK_ROWS."""
    print("[case] attn chunk refusals", flush=True)
    b = dev.zeros(1 << 18, np.float32)
    pos = dev.zeros(1, np.int32)

    def args(n, scores):
        return AttnArgs(n, 2, 1, 64, 16, 64, b.ptr, b.ptr, b.ptr, b.ptr, b.ptr, 1e-6, np.float32(0.125),
                        b.ptr, b.ptr, b.ptr, b.ptr, pos.ptr, 0, b.ptr, A8(None, None, None), scores, 0)

    for n, scores, rows in ((16, b.ptr, 0), (16, None, 4), (16, None, 16), (4, None, 4), (513, b.ptr, 64)):
        assert fused_chunk(dev)(dev.ctx, ctypes.byref(args(n, scores)), rows) == -1, (n, scores, rows)
    dev.sync()
    assert not b.numpy().any()


def widen(cache, kvt, nkv, ctx, wide, hd):
    """The cache's rows in a cache of `wide` positions per head."""
    size = (4, 2, 1)[kvt] * hd
    rows = np.zeros((nkv, wide, size), np.uint8)
    rows[:, :ctx] = cache[:nkv * ctx * size].reshape(nkv, ctx, size)
    if kvt != 2:
        return rows.ravel()
    scales = np.zeros((nkv, wide), np.float32)
    scales[:, :ctx] = cache[nkv * ctx * size:].view(np.float32).reshape(nkv, ctx)
    return np.concatenate([rows.ravel(), scales.ravel().view(np.uint8)])


@pytest.mark.parametrize("case", [
    # n, query heads, KV heads, head size, kv dtype, position of token 0
    (1, 8, 2, 256, 1, 8000), (5, 8, 2, 256, 0, 4094), (8, 4, 4, 64, 2, 250), (3, 6, 2, 128, 0, 0),
    (1, 8, 2, 256, 2, 255), (2, 8, 2, 256, 0, 511), (3, 8, 2, 256, 1, 438), (8, 8, 2, 256, 0, 1020),
    (3, 8, 2, 256, 2, 238), (5, 8, 2, 256, 1, 477), (8, 8, 2, 256, 0, 716),  # the 240-position tiles
    (8, 8, 2, 256, 0, 763), (3, 8, 2, 256, 2, 1022),  # rows of one pass and of the pipeline
], ids=lambda c: "n%d_h%d_%d_hd%d_kv%d_pos%d" % c)
def test_long_cache_equals_in_lds(dev, case):
    """A cache past 8192 positions (softmax in segments, P.V products made beside the
    chains in 256-position tiles) against the same rows in one of 8192 (attn_pv_k)."""
    n, nh, nkv, hd, kvt, pos0 = case
    print(f"[case] attn long {case}", flush=True)
    ctx, wide = 8192, 8200
    rng = np.random.default_rng(n + hd + pos0)
    ang = rng.uniform(0, 2 * np.pi, (wide, hd // 8))
    host = dict(
        q=rng.standard_normal((n, nh, 2 * hd)).astype(np.float32),
        k_in=rng.standard_normal((n, nkv * hd)).astype(np.float32),
        v_in=rng.standard_normal((n, nkv * hd)).astype(np.float32),
        q_norm=rng.uniform(0.5, 1.5, hd).astype(np.float32),
        k_norm=rng.uniform(0.5, 1.5, hd).astype(np.float32),
        cos=np.cos(ang).astype(np.float32), sin=np.sin(ang).astype(np.float32),
        kc=cache_bytes(rng, kvt, nkv, ctx, hd), vc=cache_bytes(rng, kvt, nkv, ctx, hd),
    )
    want = passes(dev, host, (n, nh, nkv, hd, ctx, kvt, pos0), 8)
    far = dict(host, **{c: widen(host[c], kvt, nkv, ctx, wide, hd) for c in ("kc", "vc")})
    got = passes(dev, far, (n, nh, nkv, hd, wide, kvt, pos0), 8)
    for k in ("o", "aq", "ad", "afs"):
        assert_bits_equal(got[k], want[k], k)
    for k in ("kc", "vc"):
        assert_bits_equal(got[k], widen(want[k], kvt, nkv, ctx, wide, hd), k)
