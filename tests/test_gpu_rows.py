"""The row kernels (passes of up to 16 rows of the layer-by-layer path) where they can go
wrong: contexts at the edges of a 64-position chunk, of the 512 positions an attention
workgroup covers, and of the 4096 positions after which a wave takes a second chunk; passes
of 1, 3 and 16 rows (the three instantiations) that cross those edges; and a captured step
replayed where more attention splits are in use than it was captured for. Logits against the
fp32 oracle (relative L2 <= 1e-2, the activations' f16 rounding), rows of one pass against
single-row passes bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

from instantllm_amd import synth, illfile as F
from oracle import illread, qwen, metrics

pytestmark = pytest.mark.gpu

REL_L2_TOL = 1e-2
VOCAB = 1024
NO_EOS = (-5, -5)
CTX = 4096 + 64


@pytest.fixture(scope="module", params=[(F.FMT_Q8, 32), (F.FMT_F16, 64)], ids=["q8g32", "f16"])
def model(request, tmp_path_factory):
    from instantllm_amd.engine import Engine
    fmt, group = request.param
    path = str(tmp_path_factory.mktemp(f"rows{fmt}") / "m.ill")
    synth.build_model(path, fmt, seed=6, shape=synth.ModelShape(layers=2, vocab=VOCAB), q8_group=group)
    m = qwen.Model(illread.load(path))
    e = Engine(path, max_context=CTX + 64, max_pass=16, max_steps=64)
    toks = [int(t) for t in np.random.default_rng(600 + fmt).integers(0, VOCAB, size=CTX)]
    e.set_state(pos=0, n=CTX, maxsteps=64, eos=NO_EOS)
    e.prefill(toks)
    yield e, m, toks, e.kv_copy_out(CTX)
    e.close()


def one(e, pos, tok):
    e.set_state(pos=pos, n=1, maxsteps=64, eos=NO_EOS)
    e.prefill([tok], write_logits=True)
    return e.read_logits(0).view(np.uint32)


@pytest.mark.parametrize("pos", [0, 55, 504, 511, 1016, 4088])
@pytest.mark.parametrize("rows", [3, 16])
def test_pass_rows_equal_single_rows(model, pos, rows):
    e, m, toks, (k, v) = model
    chain = toks[pos:pos + rows]
    singles = [one(e, pos + i, t) for i, t in enumerate(chain)]
    e.kv_copy_in(k, v)
    e.set_state(pos=pos, n=rows, maxsteps=64, eos=NO_EOS)
    e.verify_pass(rows, toks=chain, write_logits=True)
    for i in range(rows):
        assert np.array_equal(e.read_logits(i).view(np.uint32), singles[i]), (pos, rows, i)
    e.kv_copy_in(k, v)


@pytest.mark.parametrize("pos", [0, 63, 64, 511, 512, 4095, 4097])
def test_single_row_matches_oracle(model, pos):
    e, m, toks, (k, v) = model
    got = one(e, pos, toks[pos]).view(np.float32)
    e.kv_copy_in(k, v)
    cache = m.new_cache(pos + 2)
    ref = m.forward(toks[:pos + 1], cache)
    assert metrics.rel_l2(got, ref) <= REL_L2_TOL, pos


def test_captured_step_replayed_at_a_longer_context(model):
    e, m, toks, (k, v) = model
    e.set_state(pos=20, n=1, maxsteps=64, eos=NO_EOS)
    e.capture_steps(2)   # captured for one attention split
    for pos in (511, 1500, 4090):
        e.set_state(pos=pos, n=1, maxsteps=64, eos=NO_EOS)
        e.prefill([toks[pos]])
        for _ in range(2):   # two replays of two steps
            e.launch_graph(write_logits=True)
            e.sync()
        graph = e.read_logits(0).view(np.uint32)
        committed = [int(t) for t in e.out_tokens()[:5]]
        for i, t in enumerate([toks[pos]] + committed[:4]):
            last = one(e, pos + i, t)
        assert np.array_equal(last, graph), pos
        e.kv_copy_in(k, v)


@pytest.mark.parametrize("fmt", [F.FMT_Q4, F.FMT_Q8, F.FMT_F16], ids=["q4", "q8", "f16"])
def test_prompts_at_the_row_kernels_edges(fmt, tmp_path):
    """Prompts around the longest one the row kernels take (112 rows) and its 16-row groups, one
    of 513, and prompts in two calls whose second one is short (for q4 its 1, 3 and 16 rows run
    on the pass kernel): last-row logits against the oracle."""
    from instantllm_amd.engine import Engine
    path = str(tmp_path / "m.ill")
    synth.build_model(path, fmt, seed=6, shape=synth.ModelShape(layers=2, vocab=VOCAB))
    m = qwen.Model(illread.load(path))
    e = Engine(path, max_context=1024, max_pass=16, max_steps=64)
    toks = [int(t) for t in np.random.default_rng(700 + fmt).integers(0, VOCAB, size=600)]
    try:
        for parts in ((17,), (80,), (111,), (112,), (113,), (128,), (513,), (150, 16), (150, 17), (200, 97), (20, 1, 3)):
            e.set_state(pos=0, n=1, maxsteps=64, eos=NO_EOS)
            n = 0
            for k in parts:
                e.prefill(toks[n:n + k], write_logits=True)
                n += k
            ref = m.forward(toks[:n], m.new_cache(n + 1))
            assert metrics.rel_l2(e.read_logits(0), ref) <= REL_L2_TOL, parts
    finally:
        e.close()


@pytest.mark.parametrize("fmt", [F.FMT_Q4, F.FMT_F16], ids=["q4", "f16"])
def test_prompt_attention_shapes(fmt, tmp_path):
    """Both shapes of the prompt attention (chunks shared through LDS, waves per head) at the block
    counts around the switch (24 blocks of 16 rows for q4, 72 for f16), odd and even chunk counts
    and last blocks, and second calls that start inside a 64-position chunk: last-row logits
    against the oracle."""
    from instantllm_amd.engine import Engine
    path = str(tmp_path / "m.ill")
    synth.build_model(path, fmt, seed=6, shape=synth.ModelShape(layers=2, vocab=VOCAB))
    m = qwen.Model(illread.load(path))
    e = Engine(path, max_context=2176, max_pass=16, max_steps=64)
    toks = [int(t) for t in np.random.default_rng(710 + fmt).integers(0, VOCAB, size=2100)]
    cuts = ((368,), (369,), (385,), (700,), (40, 1152), (77, 1130), (1300, 750)) if fmt == F.FMT_Q4 else \
           ((1136,), (1137,), (1153,), (40, 1152), (77, 1130), (1300, 750))
    try:
        for parts in cuts:
            e.set_state(pos=0, n=1, maxsteps=64, eos=NO_EOS)
            n = 0
            for k in parts:
                e.prefill(toks[n:n + k], write_logits=True)
                n += k
            ref = m.forward(toks[:n], m.new_cache(n + 1))
            assert metrics.rel_l2(e.read_logits(0), ref) <= REL_L2_TOL, parts
    finally:
        e.close()


@pytest.mark.parametrize("graph", ["steps", "spec"])
def test_passes_queued_behind_the_contexts_end(graph, tmp_path):
    """A chain pass in the last 16 slots of the context, all of its drafts accepted, leaves the
    request finished at pos = 576 = the context; the 1- and 16-row passes of a captured graph
    that still run then change nothing, and the next request is right."""
    from instantllm_amd.engine import Engine
    path = str(tmp_path / "m.ill")
    synth.build_model(path, F.FMT_Q8, seed=6, shape=synth.ModelShape(layers=2, vocab=VOCAB))
    toks = [int(t) for t in np.random.default_rng(760).integers(0, VOCAB, size=560)]
    with Engine(path, max_context=1024, max_pass=16, max_steps=64) as big:
        big.set_state(pos=0, n=560, maxsteps=64, eos=NO_EOS)
        big.prefill(toks, write_logits=True)
        want = big.read_logits(0)
        for _ in range(16):
            big.decode_step()
        chain = [int(t) for t in big.out_tokens()[:17]]
    with Engine(path, max_context=576, max_pass=16, max_steps=64) as e:
        e.set_state(pos=0, n=560, maxsteps=64, eos=NO_EOS, tspec=16)
        (e.capture_spec if graph == "spec" else e.capture_steps)(2)
        e.prefill(toks)
        e.verify_pass(16, toks=chain[:16], write_logits=True)
        assert int(np.argmax(e.read_logits(15))) == chain[16]
        st, kv = e.get_state(), e.kv_copy_out(576)
        assert st["done"] and st["pos"] == 576
        print("finished at the context's end, launching", graph, flush=True)
        e.launch_graph()
        e.sync()
        assert e.get_state() == st
        assert all(np.array_equal(a, b) for a, b in zip(kv, e.kv_copy_out(576)))
        e.set_state(pos=0, n=560, maxsteps=64, eos=NO_EOS)
        e.prefill(toks, write_logits=True)
        assert np.array_equal(e.read_logits(0).view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("fmt", [F.FMT_Q4, F.FMT_Q8, F.FMT_F16], ids=["q4", "q8", "f16"])
def test_prompts_of_two_chunks(fmt, tmp_path):
    """Prompts past the 4096 rows of a chunk, whose last chunk has 1, 3, 16 and 17 rows: the row
    kernels' three instantiations (for q4, which runs them on its cache layout, only here) and
    their split attention states, after a chunk that computes no logits. Last-row logits and the
    decode step after them against the oracle."""
    from instantllm_amd.engine import Engine
    path = str(tmp_path / "m.ill")
    synth.build_model(path, fmt, seed=6, shape=synth.ModelShape(layers=2, vocab=VOCAB))
    m = qwen.Model(illread.load(path))
    toks = [int(t) for t in np.random.default_rng(720 + fmt).integers(0, VOCAB, size=4113)]
    cache = m.new_cache(4120)
    for c0 in range(0, 4096, 1024):   # (attention memory)
        m.forward(toks[c0:c0 + 1024], cache)
    ref = m.forward(toks[4096:], cache, all_logits=True)
    with Engine(path, max_context=4224, max_pass=16, max_steps=64) as e:
        for n in (4097, 4099, 4112, 4113):
            print("prompt", n, flush=True)
            e.set_state(pos=0, n=n, maxsteps=64, eos=NO_EOS)
            e.prefill(toks[:n], write_logits=True)
            got = e.read_logits(0)
            assert metrics.rel_l2(got, ref[n - 4097]) <= REL_L2_TOL, n
            tok = int(e.out_tokens()[0])
            assert tok == int(np.argmax(got))
            e.decode_step(write_logits=True)
            cache.len = n
            assert metrics.rel_l2(e.read_logits(0), m.forward([tok], cache)) <= REL_L2_TOL, n
            cache.len = n
            m.forward([toks[n]] if n < 4113 else [0], cache)   # the prompt's own token back in its slot
