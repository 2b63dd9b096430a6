"""GPU parity of the layer-by-layer path through the C ABI: q8 (symmetric, groups of 64 and 32) and f16
models for every pass shape, and q4 prompts longer than 16 tokens (prefill chunks on the
MFMA GEMMs). Small seeded models (3 layers, vocabulary 4096, real widths) against the fp32
oracle on the same dequantized weights. Tolerances as for q4: per-step logits relative L2
<= 1e-2, teacher-forced greedy agreement >= 99%, 1-row vs 16-row logits bit-identical.
"""
from __future__ import annotations

import numpy as np
import pytest

from instantllm_amd import synth, illfile as F
from oracle import illread, qwen, metrics, tree as T

pytestmark = pytest.mark.gpu

REL_L2_TOL = 1e-2
VOCAB = 4096
NO_EOS = (-5, -5)


def log(*a):
    print(*a, flush=True)


# q8 in the BASELINE's group of 64 and in the reference converter's own group of 32
# (Convert.swift:254-282; the engine reads the group size from the scale tensor's size)
@pytest.fixture(scope="module", params=[(F.FMT_Q8, 64), (F.FMT_Q8, 32), (F.FMT_F16, 64), (F.FMT_Q4, 64)],
                ids=["q8", "q8g32", "f16", "q4"])
def model(request, tmp_path_factory):
    from instantllm_amd.engine import Engine
    fmt, group = request.param
    path = str(tmp_path_factory.mktemp(f"fmt{fmt}g{group}") / "m.ill")
    synth.build_model(path, fmt, seed=4, shape=synth.ModelShape(layers=3, vocab=VOCAB), q8_group=group)
    log(f"engine: create small model format {fmt} group {group}")
    e = Engine(path, max_context=1024, max_pass=16, max_steps=256)
    yield fmt, e, qwen.Model(illread.load(path))
    e.close()


def test_prefill_and_decode_logits(model):
    fmt, e, m = model
    rng = np.random.default_rng(40 + fmt)
    prompt = [int(t) for t in rng.integers(0, VOCAB, size=45)]
    log(f"format {fmt}: prefill 45 + 8 decode steps")
    e.reset_out_tokens()
    e.set_state(pos=0, n=len(prompt), maxsteps=64, eos=NO_EOS)
    e.prefill(prompt, write_logits=True)
    cache = m.new_cache(128)
    ref = m.forward(prompt, cache)
    lg = e.read_logits(0)
    assert metrics.rel_l2(lg, ref) <= REL_L2_TOL
    tok = int(e.out_tokens()[0])
    assert tok == int(np.argmax(lg))
    for s in range(8):
        e.decode_step(write_logits=True)
        lg = e.read_logits(0)
        ref = m.forward([tok], cache)
        assert metrics.rel_l2(lg, ref) <= REL_L2_TOL, s
        nxt = int(e.out_tokens()[s + 1])
        assert nxt == int(np.argmax(lg))
        tok = nxt


def test_teacher_forced_agreement(model):
    fmt, e, m = model
    rng = np.random.default_rng(50 + fmt)
    prompt = [int(t) for t in rng.integers(0, VOCAB, size=20)]
    toks = e.generate(prompt, max_new=32, chunk=8)
    am, _ = m.teacher_forced(prompt, toks)
    agree, n = metrics.forced_agreement(toks, am)
    assert agree / n >= 0.99, (agree, n)


def test_tree_rows_bit_identical_to_sequential_steps(model):
    fmt, e, _ = model
    rng = np.random.default_rng(60 + fmt)
    ctx = [int(t) for t in rng.integers(0, VOCAB, size=130)]
    e.reset_out_tokens()
    e.set_state(pos=0, n=len(ctx), maxsteps=200, eos=NO_EOS)
    e.prefill(ctx)
    st = e.get_state()
    tr = synth.random_tree(rng, 16, VOCAB)
    e.set_state(pos=st["pos"], n=16, maxsteps=200, eos=NO_EOS)
    e.verify_pass(16, tree=tr, write_logits=True)
    rows = np.stack([e.read_logits(r) for r in range(16)])
    tok = tr[T.TR_TOK:T.TR_TOK + 16]
    for p in T.paths(tr):
        for k, r in enumerate(p):
            e.set_state(pos=st["pos"] + k, n=1, maxsteps=200, eos=NO_EOS)
            e.prefill([int(tok[r])], write_logits=True)
            one = e.read_logits(0)
            assert np.array_equal(one.view(np.uint32), rows[r].view(np.uint32)), (p, k, r)


def test_tree_logits_match_oracle(model):
    fmt, e, m = model
    rng = np.random.default_rng(70 + fmt)
    ctx = [int(t) for t in rng.integers(0, VOCAB, size=70)]
    e.reset_out_tokens()
    e.set_state(pos=0, n=len(ctx), maxsteps=200, eos=NO_EOS)
    e.prefill(ctx)
    st = e.get_state()
    tr = synth.random_tree(rng, 16, VOCAB)
    e.set_state(pos=st["pos"], n=16, maxsteps=200, eos=NO_EOS)
    e.verify_pass(16, tree=tr, write_logits=True)
    cache = m.new_cache(128)
    m.forward(ctx, cache)
    ref = T.tree_logits(m, cache, tr)
    for r in range(16):
        assert metrics.rel_l2(e.read_logits(r), ref[r]) <= REL_L2_TOL, r


def test_long_prefill_chunks(model):
    """A prompt of 600 tokens (one layer-by-layer chunk on the ring GEMMs), then decode. Prompts of
    several chunks: tests/test_gpu_rows.py."""
    fmt, e, m = model
    rng = np.random.default_rng(80 + fmt)
    prompt = [int(t) for t in rng.integers(0, VOCAB, size=600)]
    e.reset_out_tokens()
    e.set_state(pos=0, n=len(prompt), maxsteps=64, eos=NO_EOS)
    e.prefill(prompt, write_logits=True)
    cache = m.new_cache(640)
    ref = m.forward(prompt, cache)
    assert metrics.rel_l2(e.read_logits(0), ref) <= REL_L2_TOL
    tok = int(e.out_tokens()[0])
    e.decode_step(write_logits=True)
    assert metrics.rel_l2(e.read_logits(0), m.forward([tok], cache)) <= REL_L2_TOL


@pytest.mark.parametrize("n", [17, 31, 33, 63, 65, 511, 513])
def test_prefill_chunk_edges(model, n):
    """Prompt lengths at the edges of the prefill GEMMs' row tiles (16, 32 and 64 rows) and
    around 512, prefilled in one call and again in two calls whose second one starts
    at a position that is not a multiple of 64 (the QKV epilogue's rotary rows are read for
    pos + row): last-row logits and the first decode step after it against the oracle."""
    fmt, e, m = model
    rng = np.random.default_rng(1000 + 10 * fmt + n)
    prompt = [int(t) for t in rng.integers(0, VOCAB, size=n)]
    cache = m.new_cache(n + 8)
    ref = m.forward(prompt, cache)
    nxt = m.forward([int(np.argmax(ref))], cache)
    for split in (n, 17 + (n - 17) // 3):
        log(f"format {fmt}: prompt {n}, first call {split} rows")
        e.reset_out_tokens()
        e.set_state(pos=0, n=n, maxsteps=64, eos=NO_EOS)
        e.prefill(prompt[:split], write_logits=split == n)
        if split < n:
            e.prefill(prompt[split:], write_logits=True)
        lg = e.read_logits(0)
        assert metrics.rel_l2(lg, ref) <= REL_L2_TOL, split
        tok = int(e.out_tokens()[e.get_state()["step"] - 1])   # the last call's token
        assert tok == int(np.argmax(lg))
        if tok != int(np.argmax(ref)):   # a near tie in the logits: the step would differ
            continue
        e.decode_step(write_logits=True)
        assert metrics.rel_l2(e.read_logits(0), nxt) <= REL_L2_TOL, split


def test_split_attention_rows_bit_identical_long_context(tmp_path):
    """Past 1024 positions the 1-row and 16-row attention of the layer-by-layer path is split
    over several workgroups per (row, head). The split follows the launch (1-row steps here
    run both split and unsplit) but the grouping of the arithmetic follows the row alone, so
    tree rows must still equal sequential 1-row steps bit for bit, and match the oracle."""
    from instantllm_amd.engine import Engine
    path = str(tmp_path / "m.ill")
    synth.build_model(path, F.FMT_Q8, seed=4, shape=synth.ModelShape(layers=3, vocab=VOCAB))
    m = qwen.Model(illread.load(path))
    e = Engine(path, max_context=2048, max_pass=16, max_steps=256)
    try:
        rng = np.random.default_rng(91)
        ctx = [int(t) for t in rng.integers(0, VOCAB, size=1015)]
        e.reset_out_tokens()
        e.set_state(pos=0, n=len(ctx), maxsteps=200, eos=NO_EOS)
        log("q8: prefill 1015, 16-row tree pass, sequential steps along its paths")
        e.prefill(ctx)
        st = e.get_state()
        tr = synth.random_tree(rng, 16, VOCAB)
        e.set_state(pos=st["pos"], n=16, maxsteps=200, eos=NO_EOS)
        e.verify_pass(16, tree=tr, write_logits=True)
        rows = np.stack([e.read_logits(r) for r in range(16)])
        cache = m.new_cache(1100)
        m.forward(ctx, cache)
        ref = T.tree_logits(m, cache, tr)
        for r in range(16):
            assert metrics.rel_l2(rows[r], ref[r]) <= REL_L2_TOL, r
        tok = tr[T.TR_TOK:T.TR_TOK + 16]
        for p in T.paths(tr)[:3]:
            for k, r in enumerate(p):
                e.set_state(pos=st["pos"] + k, n=1, maxsteps=200, eos=NO_EOS)
                e.prefill([int(tok[r])], write_logits=True)
                one = e.read_logits(0)
                assert np.array_equal(one.view(np.uint32), rows[r].view(np.uint32)), (p, k, r)
    finally:
        e.close()
