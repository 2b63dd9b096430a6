"""q4 1-row steps past 512 positions, where other workgroups evaluate the attention chunks that
a head's own workgroup has no wave for: contexts at the edges of the chunks, of the rounds of
eight chunks and of the helpers' second round (from 88 chunks), against the rows of a 16-row
chain pass (whose attention workgroups evaluate every chunk themselves) bit for bit, stepped
one by one and replayed from a captured graph."""
from __future__ import annotations

import numpy as np
import pytest

from instantllm_amd import synth, illfile as F

pytestmark = pytest.mark.gpu

VOCAB = 1024
NO_EOS = (-5, -5)
CTX = 6016


@pytest.fixture(scope="module")
def engine(tmp_path_factory):
    from instantllm_amd.engine import Engine
    path = str(tmp_path_factory.mktemp("long") / "m.ill")
    synth.build_model(path, F.FMT_Q4, seed=8, shape=synth.ModelShape(layers=3, vocab=VOCAB), quantizer="minmax")
    e = Engine(path, max_context=CTX, max_pass=16, max_steps=64)
    rng = np.random.default_rng(8)
    kv = [rng.standard_normal((3, 2, CTX, 64), dtype=np.float32).astype(np.float16).view(np.uint16) for _ in range(2)]
    yield e, kv
    e.close()


@pytest.mark.parametrize("pos", [448, 504, 511, 512, 513, 575, 576, 633, 1016, 1024, 2111, 4095, 5200, 5630, 5700, 5900])
def test_steps_equal_chain_rows(engine, pos):
    e, (k, v) = engine
    print("pos", pos, flush=True)
    toks = [int(t) for t in np.random.default_rng(pos).integers(0, VOCAB, size=16)]
    e.kv_copy_in(k, v)
    singles = []
    for i, t in enumerate(toks):
        e.set_state(pos=pos + i, n=1, maxsteps=64, eos=NO_EOS)
        e.prefill([t], write_logits=True)
        singles.append(e.read_logits(0).view(np.uint32))
    e.kv_copy_in(k, v)
    e.set_state(pos=pos, n=16, maxsteps=64, eos=NO_EOS)
    e.verify_pass(16, toks=toks, write_logits=True)
    for i in range(16):
        assert np.isfinite(singles[i].view(np.float32)).all()
        assert np.array_equal(e.read_logits(i).view(np.uint32), singles[i]), (pos, i)


def test_graph_replays_cross_the_edge(engine):
    """A graph of steps captured below 512 positions and replayed across it equals single steps."""
    e, (k, v) = engine
    e.kv_copy_in(k, v)
    e.set_state(pos=500, n=1, maxsteps=64, eos=NO_EOS)
    e.prefill([5])
    for _ in range(20):
        e.decode_step(write_logits=True)
    want, lg = e.out_tokens()[:21].copy(), e.read_logits(0).view(np.uint32)
    e.kv_copy_in(k, v)
    e.set_state(pos=500, n=1, maxsteps=64, eos=NO_EOS)
    e.prefill([5])
    e.capture_steps(10)
    for _ in range(2):
        e.launch_graph(write_logits=True)
        e.sync()
    assert np.array_equal(e.out_tokens()[:21], want)
    assert np.array_equal(e.read_logits(0).view(np.uint32), lg)
