"""GPU parity of the DeltaNet chunk kernels (more than 8 tokens, no log: conv, norms and gates with
the tokens in parallel, then kv chains and skewed o chains in waves of their own).

The recurrence is compared with the oracle and the whole mixer with lin_mix_k, the one-launch kernel
that takes the same pass under capture. Bar: bit-exact for outputs, recurrent state and conv state.
Sizes at the pipeline's edges: 9 tokens (less than the 15 steps a sum takes), 16 and 17 (two batches
of 8, one more token), 48, 63, 64 (the 8 batches that the ring holds), 209 and 512 (the ring wraps),
pending replays, shared key heads, dk 64 to 256, a last column group that is not 16 wide."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

import oracle
from nibblemac_amd.nmx import A8, LinArgs, LinMixArgs, LinPreArgs
from tests.refmath import state_from_dev, state_to_dev
from tests.test_gpu_linmix import make_case, p, run
from tests.test_gpu_q4k import assert_bits_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("case", [
    # n, heads, rep, dk, dv, keep
    (9, 2, 1, 128, 128, 0), (16, 2, 1, 128, 128, 3), (17, 4, 2, 128, 64, 0), (48, 2, 1, 64, 64, 9),
    (63, 2, 1, 256, 32, 1), (64, 16, 1, 128, 128, 0), (64, 3, 3, 64, 24, 0), (31, 2, 1, 128, 8, 5),
], ids=lambda c: "n%d_h%d_rep%d_dk%d_dv%d_keep%d" % c)
def test_rule_equals_oracle(dev, case):
    n, heads, rep, dk, dv, keep = case
    print(f"[case] lin chunk rule {case}", flush=True)
    rng = np.random.default_rng(n + dk + dv + keep)
    kd, stride = heads // rep * dk, 2 * (heads // rep) * dk + heads * dv
    qkv = rng.standard_normal((n, stride)).astype(np.float32)
    qkv[:, :2 * kd] *= np.float32(dk ** -0.5)
    decay = rng.uniform(0.8, 1.0, (n, heads)).astype(np.float32)
    beta = rng.uniform(0.1, 0.9, (n, heads)).astype(np.float32)
    S = (rng.standard_normal((heads, dk, dv)) * 0.05).astype(np.float32)
    S.ravel()[::7] = -0.0
    pend = (rng.standard_normal((max(keep, 1), heads, dk + dv + 1)) * 0.1).astype(np.float32)
    want_S, want_o, _ = oracle.lin_rule(qkv, decay, beta, S, n=n, heads=heads, rep=rep, dk=dk, dv=dv,
                                        pend=pend, keep=keep)
    dS, dq, dd, db = (dev.to_device(x) for x in (state_to_dev(S, heads, dk, dv), qkv, decay, beta))
    o, dp = dev.zeros((n, heads * dv), np.float32), dev.to_device(pend)
    dev.lin_rule(n=n, heads=heads, rep=rep, dk=dk, dv=dv, qkv_stride=stride, o_stride=heads * dv,
                 qkv=dq, decay=dd, beta=db, S=dS, o=o, pend=dp, keep=keep)
    dev.sync()
    assert_bits_equal(o.numpy(), want_o, "o")
    assert_bits_equal(state_from_dev(dS.numpy(), heads, dk, dv), want_S, "state")


def chunk_fn(dev):
    fn = dev.lib.nmx_lin_mix_chunk
    fn.restype, fn.argtypes = ctypes.c_int, [ctypes.c_void_p, ctypes.POINTER(LinMixArgs)]
    return fn


def one_launch(dev, c):
    """The pass through lin_mix_k: a captured launch, which does not use the context's workspace."""
    n, heads, dk, dv, C = (c[k] for k in ("n", "heads", "dk", "dv", "C"))
    d = {k: dev.to_device(v) for k, v in c["host"].items()}
    nb = heads * dv // 32
    y = dev.zeros((n, heads * dv), np.float32)
    aq, ad, afs = (dev.zeros((nb, n, 32), np.int8), dev.zeros((nb, n), np.float32),
                   dev.zeros((nb, n), np.float32))
    pre = LinPreArgs(n, C, c["K"], dk, c["kd"], p(d["raw"]), C, None, p(d["state"]), p(d["conv_w"]),
                     None, np.float32(1.0 / np.sqrt(dk)), 1e-6, p(d["b"]), p(d["a"]), heads, heads,
                     p(d["A_log"]), None, p(d["dt_bias"]), None, None)
    rule = LinArgs(n, heads, 1, dk, dv, C, heads * dv, None, None, None, p(d["S"]), None, None,
                   p(d["pend"]), c["keep"], 0, None)
    dev.graph_begin()
    dev.lin_mix(LinMixArgs(pre, rule, p(d["z"]), heads * dv, p(d["norm_w"]), 1e-6, p(y), heads * dv,
                           A8(p(aq), p(ad), p(afs))))
    g = dev.graph_end()
    dev.graph_launch(g)
    dev.sync()
    dev.graph_destroy(g)
    return dict(aq=aq.numpy(), ad=ad.numpy(), afs=afs.numpy(), y=y.numpy(), S=d["S"].numpy(),
                state=d["state"].numpy())


@pytest.mark.parametrize("case", [
    # n, heads, dk, dv, keep
    (9, 4, 128, 128, 0), (13, 4, 128, 128, 4), (33, 4, 64, 64, 0), (64, 16, 128, 128, 0),
    (57, 2, 64, 128, 2),
], ids=lambda c: "n%d_h%d_dk%d_dv%d_keep%d" % c)
def test_mixer_equals_one_launch(dev, case):
    n, heads, dk, dv, keep = case
    print(f"[case] lin chunk mixer {case}", flush=True)
    rng = np.random.default_rng(3 * n + heads + dk + keep)
    c = make_case(dev, rng, n, heads, 1, dk, dv, logged=False, keep=keep)
    want = one_launch(dev, c)
    got = run(dev, c, fused=True)
    for k in want:
        assert_bits_equal(got[k], want[k], k)


@pytest.mark.parametrize("case", [
    # n, heads, rep, dk, dv, keep
    (257, 2, 1, 256, 64, 3), (256, 4, 2, 128, 32, 0), (273, 2, 1, 64, 64, 0), (512, 2, 2, 128, 32, 0),
    (209, 2, 1, 128, 32, 2),
], ids=lambda c: "n%d_h%d_rep%d_dk%d_dv%d_keep%d" % c)
def test_long_chunk_equals_pieces(dev, case):
    """nmx_lin_mix_chunk above 64 rows (batches of 8 up to 256 tokens, of 16 above) against passes of
    64 over the same rows, the states carried from one to the next."""
    n, heads, rep, dk, dv, keep = case
    print(f"[case] lin long chunk {case}", flush=True)
    fn = chunk_fn(dev)
    c = make_case(dev, np.random.default_rng(n + dk), n, heads, rep, dk, dv, logged=False, keep=keep)
    h, C, vd = c["host"], c["C"], heads * dv

    def passes(step):
        d = {k: dev.to_device(h[k]) for k in ("A_log", "dt_bias", "conv_w", "state", "S", "pend", "norm_w")}
        ys = []
        for t0 in range(0, n, step):
            m = min(step, n - t0)
            x = {k: dev.to_device(h[k][t0:t0 + m]) for k in ("raw", "z", "b", "a")}
            conv, o, y = (dev.zeros((m, w), np.float32) for w in (C, vd, vd))
            beta, decay = (dev.zeros((m, heads), np.float32) for _ in range(2))
            pre = LinPreArgs(m, C, c["K"], dk, c["kd"], p(x["raw"]), C, p(conv), p(d["state"]),
                             p(d["conv_w"]), None, np.float32(1.0 / np.sqrt(dk)), 1e-6, p(x["b"]),
                             p(x["a"]), heads, heads, p(d["A_log"]), None, p(d["dt_bias"]), p(beta),
                             p(decay))
            rule = LinArgs(m, heads, rep, dk, dv, C, vd, p(conv), p(decay), p(beta), p(d["S"]), p(o),
                           None, p(d["pend"]), keep if t0 == 0 else 0, 0, None)
            dev.check(fn(dev.ctx, ctypes.byref(LinMixArgs(pre, rule, p(x["z"]), vd, p(d["norm_w"]), 1e-6,
                                                          p(y), vd, A8(None, None, None)))))
            dev.sync()
            ys.append(y.numpy())
        return np.concatenate(ys), d["S"].numpy(), d["state"].numpy()

    for got, want, what in zip(passes(512), passes(64), ("y", "state", "conv state")):
        assert_bits_equal(got, want, what)


def buffers(dev, c, fill):
    """The mixer's arguments of nmx_lin_mix_chunk, every intermediate buffer filled with `fill`."""
    n, heads, rep, dk, dv, C = c["n"], c["heads"], c["rep"], c["dk"], c["dv"], c["C"]
    d, vd = {k: dev.to_device(v) for k, v in c["host"].items()}, heads * dv
    mid = {k: dev.to_device(np.full((n, w), fill, np.float32))
           for k, w in (("out", C), ("beta", heads), ("decay", heads), ("o", vd))}
    y = dev.zeros((n, vd), np.float32)
    pre = LinPreArgs(n, C, c["K"], dk, c["kd"], p(d["raw"]), C, p(mid["out"]), p(d["state"]),
                     p(d["conv_w"]), None, np.float32(1.0 / np.sqrt(dk)), 1e-6, p(d["b"]), p(d["a"]),
                     heads, heads, p(d["A_log"]), None, p(d["dt_bias"]), p(mid["beta"]), p(mid["decay"]))
    rule = LinArgs(n, heads, rep, dk, dv, C, vd, p(mid["out"]), p(mid["decay"]), p(mid["beta"]),
                   p(d["S"]), p(mid["o"]), None, p(d["pend"]), c["keep"], 0, None)
    args = LinMixArgs(pre, rule, p(d["z"]), vd, p(d["norm_w"]), 1e-6, p(y), vd, A8(None, None, None))
    return args, d, mid, y


@pytest.mark.parametrize("n,keep", [(9, 0), (64, 3)])
def test_mixer_leaves_buffers_untouched(dev, n, keep):
    """nmx_lin_mix in the fused kernel's shapes does not use the caller's intermediate buffers, and the
    results of two passes in a row (the context's workspace holds the first one's) are lin_mix_k's."""
    print(f"[case] lin chunk mixer buffers n={n} keep={keep}", flush=True)
    c = make_case(dev, np.random.default_rng(n + keep), n, 4, 1, 128, 128, logged=False, keep=keep)
    want = one_launch(dev, c)
    for _ in range(2):
        args, d, mid, y = buffers(dev, c, -7.0)
        dev.lin_mix(args)
        dev.sync()
        for k, b in mid.items():
            assert (b.numpy() == -7.0).all(), f"{k} written"
        for got, k in ((y, "y"), (d["S"], "S"), (d["state"], "state")):
            assert_bits_equal(got.numpy(), want[k], k)


@pytest.mark.parametrize("n", [9, 64])
def test_overlapping_buffers_take_one_launch(dev, n):
    """nmx_lin_mix_chunk of at most 64 rows whose o lies in the raw inputs: lin_mix_k, or the chunk
    kernels over the context's workspace; the same bits, and the raw inputs untouched."""
    print(f"[case] lin chunk mixer overlap n={n}", flush=True)
    c = make_case(dev, np.random.default_rng(n), n, 4, 1, 128, 128, logged=False)
    want = one_launch(dev, c)
    args, d, mid, y = buffers(dev, c, 0.0)
    args.rule.o = p(d["raw"])
    dev.check(chunk_fn(dev)(dev.ctx, ctypes.byref(args)))
    dev.sync()
    assert_bits_equal(d["raw"].numpy(), c["host"]["raw"], "raw inputs")
    for got, k in ((y, "y"), (d["S"], "S"), (d["state"], "state")):
        assert_bits_equal(got.numpy(), want[k], k)


def test_long_chunk_refusals(dev):
    """Above 64 rows nmx_lin_mix_chunk refuses on the host what only the other kernels take; n is
    also bounded by NMX_CHUNK_ROWS, and by 64 in nmx_lin_mix."""
    print("[case] lin chunk refusals", flush=True)
    c = make_case(dev, np.random.default_rng(1), 65, 2, 1, 128, 128, logged=False)
    log = dev.zeros((65, 2, 257), np.float32)

    def change(args, d, mid, what):
        if what == "log":
            args.rule.log = p(log)
        elif what == "no o":
            args.rule.o = None
        elif what == "o in raw":
            args.rule.o = p(d["raw"])
        elif what == "qkv elsewhere":
            args.rule.qkv = p(d["raw"])
        elif what == "513 rows":
            args.pre.n = args.rule.n = 513

    for what in ("log", "no o", "o in raw", "qkv elsewhere", "513 rows"):
        args, d, mid, y = buffers(dev, c, 0.0)
        change(args, d, mid, what)
        assert chunk_fn(dev)(dev.ctx, ctypes.byref(args)) == -1, what
        assert b"nmx_lin_mix" in dev.lib.nmx_error(dev.ctx)
        dev.sync()
        assert_bits_equal(d["S"].numpy(), c["host"]["S"], "state")
    args, d, mid, y = buffers(dev, c, 0.0)
    assert dev.lib.nmx_lin_mix(dev.ctx, ctypes.byref(args)) == -1
