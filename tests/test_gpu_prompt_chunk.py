"""A prompt's forward passes of up to 512 rows against the same prompt fed in pieces of at most 64
(passes of 64 rows or fewer, which the other GPU tests pin): the last token's logits and the whole
state (conv and recurrent states, KV rows) bit for bit, and the tokens and state of a speculative
generation behind the prompt (its prefill also runs the MTP head over the chunk's rows). Lengths at
the edges: one row past 64, one past the attention's slice of 256 rows, one past a full chunk; the
three cache formats; a context shorter than a chunk."""
from __future__ import annotations

from dataclasses import replace

import numpy as np
import pytest

from nibblemac_amd import pqfile
from nibblemac_amd.pinfer import Model
from tests.test_gpu_q4k import assert_bits_equal

pytestmark = pytest.mark.gpu

SHAPES = {"small": pqfile.SMALL,                               # shared key heads, dk = 64
          "wide": replace(pqfile.SMALL, lin_k_heads=4, lin_k_dim=128, lin_v_dim=128,
                         head_dim=256, rot=64)}


@pytest.fixture(scope="module")
def models(tmp_path_factory):
    d = tmp_path_factory.mktemp("chunk")
    return {k: pqfile.write_model(d / f"{k}.pq", s, seed=3, random_norms=True)
            for k, s in SHAPES.items()}


@pytest.mark.parametrize("shape,n,kv,ctx", [("small", 65, 0, 1024), ("small", 320, 1, 1024),
                                            ("wide", 257, 0, 512), ("wide", 513, 2, 640),
                                            ("small", 100, 0, 100)])
def test_prompt_equals_pieces(models, shape, n, kv, ctx):
    print(f"[case] prompt chunk {shape} n={n} kv={kv} ctx={ctx}", flush=True)
    prompt = np.random.default_rng(n).integers(0, SHAPES[shape].vocab, n)
    with Model(models[shape], max_ctx=ctx, kv_dtype=kv) as m:
        got = m.eval(prompt)
        got_state = m.state_save()
        m.reset()
        for t in range(0, n, 64):
            want = m.eval(prompt[t:t + 64])
        assert_bits_equal(got, want, "logits")
        assert got_state == m.state_save()


@pytest.mark.parametrize("shape,n", [("small", 130), ("wide", 300)])
def test_generation_behind_prompt(models, shape, n):
    print(f"[case] prompt chunk generation {shape} n={n}", flush=True)
    prompt = np.random.default_rng(7 * n).integers(0, SHAPES[shape].vocab, n)
    with Model(models[shape], max_ctx=640) as m:
        tokens, stats = m.generate(prompt, 12, k=3, draft_vocab=512)
        state = m.state_save()
        m.reset()
        for t in range(0, n - 1, 64):  # the prompt but its last token, then the generation on it
            m.eval(prompt[t:min(t + 64, n - 1)], logits=False)
        again, _ = m.generate(prompt[-1:], 12, k=3, draft_vocab=512, cont=True)
        plain, _ = m.generate(prompt, 12)
        assert tokens == again == plain
        m.reset()
        assert m.generate(prompt, 12, k=3, draft_vocab=512)[0] == tokens and m.state_save() == state
