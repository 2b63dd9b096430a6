"""Attention keeps fp32's precision in queries and probabilities (q8 / f16 passes of up to 16 rows,
prompts of all formats): caches on which operands of 16 bits, or pairs of them whose low halves
run into f16's subnormals, show in the logits. The attention norm of layer 0 is set to zero, so that
q is the QKV bias (fp32, no activation rounding) and the rows' own keys and values are zero; keys and
values are written into the cache. Logits against the oracle in float64, relative L2 <= 1.5e-3: the
f16 roundings of the attention output, of the MLP's input and of its hidden units (2^-12 each, rms
1.4e-4) leave 3e-4 to 6e-4. (Pairs of unscaled values: 1.7e-3 to 9e-3.)"""
from __future__ import annotations

import struct

import numpy as np
import pytest

from instantllm_amd import illfile as F, synth
from oracle import illread, metrics, qwen

pytestmark = pytest.mark.gpu
VOCAB, CTX, NO_EOS = 1024, 2176, (-5, -5)
REL_L2_TOL = 1.5e-3


@pytest.fixture(scope="module", params=[F.FMT_Q8, F.FMT_F16], ids=["q8", "f16"])
def base(request, tmp_path_factory):
    path = str(tmp_path_factory.mktemp("att") / "m.ill")
    synth.build_model(path, request.param, seed=9, shape=synth.ModelShape(layers=1, vocab=VOCAB))
    return path


def patched(base, tmp_path, bq):
    """The model with ln1 = 0 and the QKV bias (bq, 0, 0)."""
    path = str(tmp_path / "p.ill")
    data = bytearray(open(base, "rb").read())
    count = struct.unpack_from("<I", data, 12)[0]
    tab = np.frombuffer(bytes(data[16:16 + 16 * count]), "<u8").reshape(count, 2)
    bias = np.concatenate([bq.reshape(-1), np.zeros(256)])[F.qkv_row_order()].astype("<f4").tobytes()
    for tid, val in ((F.layer_id(0, F.ATTN_NORM), bytes(4 * 896)), (F.layer_id(0, F.BQKV), bias)):
        off, size = (int(x) for x in tab[tid])
        assert size == len(val)
        data[off:off + size] = val
    open(path, "wb").write(data)
    return path


def check(path, pos, k, v):
    """k, v: f16 [2, pos, 64]. The logits of one row at pos against the float64 oracle."""
    from instantllm_amd.engine import Engine
    m = qwen.Model(illread.load(path), dtype=np.float64)
    cache = m.new_cache(pos + 1)
    cache.k[0][:, :pos], cache.v[0][:, :pos], cache.len = k, v, pos
    ref = m.forward([7], cache)
    with Engine(path, max_context=CTX, max_pass=16, max_steps=16) as e:
        e.kv_copy_in(k[None].view(np.uint16), v[None].view(np.uint16))
        e.set_state(pos=pos, n=1, maxsteps=16, eos=NO_EOS)
        e.prefill([7], write_logits=True)
        got = e.read_logits(0)
    err = metrics.rel_l2(got, ref)
    print("rel_l2", err, flush=True)
    assert err <= REL_L2_TOL


def check_prompt(path, k, v, rows, rng):
    """k, v: f16 [2 layers, 2, 300, 64]. The last row's logits of a prompt of `rows` tokens after them."""
    from instantllm_amd.engine import Engine
    m = qwen.Model(illread.load(path), dtype=np.float64)
    cache = m.new_cache(300 + rows)
    for l in range(2):
        cache.k[l][:, :300], cache.v[l][:, :300] = k[l], v[l]
    cache.len = 300
    toks = [int(t) for t in rng.integers(0, VOCAB, size=rows)]
    ref = m.forward(toks, cache)
    with Engine(path, max_context=CTX, max_pass=16, max_steps=16) as e:
        e.kv_copy_in(k.view(np.uint16), v.view(np.uint16))
        e.set_state(pos=300, n=rows, maxsteps=16, eos=NO_EOS)
        e.prefill(toks, write_logits=True)
        err = metrics.rel_l2(e.read_logits(0), ref)
    print("rel_l2", err, flush=True)
    assert err <= REL_L2_TOL


def rope(x, pos):
    c, s = qwen.rope_cos_sin(np.array([pos]), np.float64)
    return x * c + qwen.rotate_half(x) * s


@pytest.mark.parametrize("pos", [300, 700, 2100])
def test_small_probabilities_beside_a_sink(base, tmp_path, pos):
    """One key takes nearly all of the weight and has no value; the output is the sum of the
    chunk's other probabilities of 2^-19 to 2^-21 (a level per head) times large values."""
    rng = np.random.default_rng(pos)
    u = rng.standard_normal(64)
    level = 19 + 2 * np.arange(14) / 13
    bq = u[None] * level[:, None] / level.mean()
    r = rope(u, pos)[0]
    k = np.zeros((2, pos, 64), np.float16)
    k[:, 3] = (r * 8 * level.mean() * np.log(2) / (r @ r)).astype(np.float16)
    v = np.broadcast_to((3e4 * rng.uniform(-1, 1, size=(2, 1, 64))).astype(np.float16), k.shape).copy()
    v[:, 3], v[:, 64:] = 0, 0   # (another chunk's probabilities are relative to its own largest)
    check(patched(base, tmp_path, bq), pos, k, v)


@pytest.mark.parametrize("pos", [300, 700, 2100])
def test_small_queries_against_large_keys(base, tmp_path, pos):
    rng = np.random.default_rng(pos)
    bq = 1.5e-4 * rng.standard_normal((14, 64))
    k = (6e4 * rng.uniform(-1, 1, size=(2, pos, 64))).astype(np.float16)
    v = rng.standard_normal((2, pos, 64)).astype(np.float16)
    check(patched(base, tmp_path, bq), pos, k, v)


@pytest.mark.parametrize("pos", [300, 700])
def test_large_queries_against_small_keys(base, tmp_path, pos):
    """q / 8 beyond f16's range."""
    rng = np.random.default_rng(pos)
    bq = 1e6 * rng.standard_normal((14, 64))
    k = (2e-5 * rng.uniform(-1, 1, size=(2, pos, 64))).astype(np.float16)
    v = rng.standard_normal((2, pos, 64)).astype(np.float16)
    check(patched(base, tmp_path, bq), pos, k, v)


@pytest.mark.parametrize("scale", [1e-4, 4e5])
@pytest.mark.parametrize("fmt,rows", [(F.FMT_Q4, 400), (F.FMT_F16, 150)])
def test_prompt_queries_small_and_large(tmp_path, fmt, rows, scale):
    """Prompts with queries of 1e-4 and 4e5, the keys' size inverse."""
    rng = np.random.default_rng(rows)
    path = str(tmp_path / "m.ill")
    synth.build_model(path, fmt, seed=9, shape=synth.ModelShape(layers=2, vocab=VOCAB))
    path = patched(path, tmp_path, scale * rng.uniform(-1, 1, size=(14, 64)))
    k, v = rng.uniform(-1, 1, size=(2, 2, 2, 300, 64))
    check_prompt(path, (6 / scale * k).astype(np.float16), v.astype(np.float16), rows, rng)


@pytest.mark.parametrize("fmt,rows", [(F.FMT_Q4, 400), (F.FMT_Q4, 40), (F.FMT_F16, 1200), (F.FMT_F16, 150)])
def test_prompt_chunks_far_below_the_largest_score(tmp_path, fmt, rows):
    """Prompts on both shapes of the prompt attention (two layers, so that layer 0 runs for every
    row): the first chunk holds a key that takes nearly all of the weight and no values, the
    chunks after it probabilities of 2^-19 to 2^-21 and large values. q lies in dims that the
    rotary embedding hardly turns, so that this holds for every row."""
    path = str(tmp_path / "m.ill")
    synth.build_model(path, fmt, seed=9, shape=synth.ModelShape(layers=2, vocab=VOCAB))
    rng = np.random.default_rng(rows)
    pos = 300
    u = np.zeros(64)
    u[24:32], u[56:] = rng.standard_normal(8), rng.standard_normal(8)
    level = 19 + 2 * np.arange(14) / 13
    path = patched(path, tmp_path, u[None] * level[:, None] / level.mean())
    r = rope(u, pos)[0]
    k, v = np.zeros((2, 2, 2, pos, 64), np.float16)
    k[0, :, 3] = (r * 8 * level.mean() * np.log(2) / (r @ r)).astype(np.float16)
    v[0, :, 64:] = (3e4 * rng.uniform(-1, 1, size=(2, 1, 64))).astype(np.float16)
    check_prompt(path, k, v, rows, rng)
