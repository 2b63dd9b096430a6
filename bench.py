"""Benchmark of the MI355X decode hot path (BASELINE.json metric).

Workload ("config 2"): the full Qwen2.5-0.5B-shaped q4 model
(24 layers, vocabulary 151936, affine group-64 4-bit weights) generated from seed 2; a
256-position prefix K/V cache prefilled from random prompt tokens; then `--steps` greedy
1-row decode steps, each one persistent-kernel launch, all recorded in one hipGraph.
Inputs are resident in HBM before timing starts. Also timed: the 16-row tree-verify pass
of config 3 (seed 3, prefix 512).

A step is one pass of the hot path over one token. value = tokens/s of the timed steps;
the line also carries us_per_token, the roofline of the dominant kernel (the pass kernel
is the whole step) and the CPU baseline (numpy fp32 oracle on the same dequantized
weights, rank 0 only, bounded sample).

Usage: python bench.py [--gpus 1] [--steps 64] [--warmup 8] [--no-cpu]
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time
from pathlib import Path

# BLAS threads of the CPU baseline, fixed before numpy loads its BLAS: the host's CPU share
# (OMP_NUM_THREADS where the environment sets it, else the cores this process may run on),
# the same count for OpenBLAS and MKL.
CPU_THREADS = int(os.environ.get("OMP_NUM_THREADS") or len(os.sched_getaffinity(0)) or 1)
for _v in ("OMP_NUM_THREADS", "OPENBLAS_NUM_THREADS", "MKL_NUM_THREADS"):
    os.environ.setdefault(_v, str(CPU_THREADS))

import numpy as np  # noqa: E402

ROOT = Path(__file__).resolve().parent
sys.path.insert(0, str(ROOT))

METRIC = json.loads((ROOT / "BASELINE.json").read_text())["metric"] if (ROOT / "BASELINE.json").exists() else \
    "q4 decode us/token (1 row) + achieved HBM GB/s vs peak; 16-row verify us"
HBM_PEAK_GBS = 8000.0
Q4_MATRIX_BYTES = 277_853_184     # q4 codes + scales of every matrix incl. the tied lm_head
F32_NORM_BIAS_BYTES = 286_208     # f32 norms + QKV biases as stored in .ill v1
EMBED_ROW_BYTES = 504             # one q4 embedding row (448 B codes + 56 B scales)
KV_BYTES_PER_POS = 12_288         # 24 layers x 2 KV heads x (K + V) x 64 x 2 B
# HBM bytes per launch of ill_pass_kernel<1> measured with rocprofv3 FETCH_SIZE and
# WRITE_SIZE (one counter per run, median over single dispatches), each scaled by the
# reading of a plain 256 MiB device copy (fetch x 2.000, write x 1.000):
# (162,670.1 x 2 + 16,358.2) KiB, measured on the pass kernel of commit 12e9d07.
# Source and commands: profiles/pass_kernel_q4_decode_config2.md
TRAFFIC_BYTES_PER_STEP = 349_899_200
# MFMA utilisation of the pass kernels (commit 12e9d07) and of the prefill kernels (commit
# 89bb7e2), from rocprofv3 SQ_VALU_MFMA_BUSY_CYCLES over the kernel durations
# (profiles/pass_kernel_q4_decode_config2.md, profiles/layer_by_layer_q8_f16_config4.md)
MFMA_COUNTERS = {
    "ill_pass_kernel<16> (16-row verify)": {"mfma_busy": 0.0111, "int8_TOPs": 48.1},
    "ill_pass_kernel<1> (1-row step)": {"mfma_busy": 0.0122, "int8_TOPs": 54.8},
    "prefill gate/up GEMM (f16, 512 rows)": {"mfma_busy": 0.184, "f16_TFLOPs": 463},
    "prefill O GEMM (f16, 512 rows)": {"mfma_busy": 0.048, "f16_TFLOPs": 120},
    "prefill down GEMM (f16, 512 rows)": {"mfma_busy": 0.143, "f16_TFLOPs": 359},
    "prefill QKV GEMM (f16, 512 rows)": {"mfma_busy": 0.039, "f16_TFLOPs": 97},
    "prefill attention (512 rows, q8 / f16)": {"mfma_busy": 0.058, "f16_TFLOPs": 146},
}


def step_bytes(L: float) -> float:
    """Algorithmic HBM bytes of one 1-row q4 step attending to L positions."""
    return Q4_MATRIX_BYTES + F32_NORM_BIAS_BYTES + EMBED_ROW_BYTES + KV_BYTES_PER_POS * L + KV_BYTES_PER_POS


def model_path(fmt: int, seed: int) -> str:
    from instantllm_amd import synth
    return synth.cached_model(fmt, seed)


def blas_vendor() -> str:
    """numpy's BLAS as numpy.show_config reports it."""
    try:
        cfg = np.show_config(mode="dicts")
        b = cfg.get("Build Dependencies", {}).get("blas", {})
        return f"{b.get('name', '?')} {b.get('version', '')}".strip()
    except Exception as exc:   # older numpy: no dict mode
        return f"unknown ({type(exc).__name__})"


def cpu_baseline(n_decode: int = 32) -> dict:
    """The numpy fp32 oracle on the config-0 model (full f16, seed 0, dequantized to fp32):
    the 48-token prefill, then `n_decode` greedy decode steps; median and min step time."""
    from instantllm_amd import synth, illfile as F
    from oracle import illread, qwen
    path = synth.cached_model(F.FMT_F16, 0)
    m = qwen.Model(illread.load(path))
    prompt = [int(t) for t in np.random.default_rng(0).integers(0, F.VOCAB, size=48)]
    cache = m.new_cache(len(prompt) + n_decode + 1)
    t0 = time.perf_counter()
    lg = m.forward(prompt, cache)
    t1 = time.perf_counter()
    times = []
    tok = int(np.argmax(lg))
    for _ in range(n_decode):
        s = time.perf_counter()
        lg = m.forward([tok], cache)
        times.append(time.perf_counter() - s)
        tok = int(np.argmax(lg))
    med = float(np.median(times))
    return {
        "value": round(1.0 / med, 3), "unit": "tok/s", "cores": CPU_THREADS, "kind": "port",
        "blas": blas_vendor(),
        "prefill48_ms": round((t1 - t0) * 1e3, 2),
        "cpu_ms_per_token_median": round(med * 1e3, 3), "cpu_ms_per_token_min": round(min(times) * 1e3, 3),
        "sample": f"config 0: numpy fp32 oracle (oracle/qwen.py) on the dequantized f16 seed-0 model "
                  f"(24 layers, vocab 151936, 1.98 GB fp32), 48-token prefill {(t1 - t0) * 1e3:.0f} ms, then "
                  f"{n_decode} greedy decode steps, median {med * 1e3:.1f} ms (min {min(times) * 1e3:.1f} ms); "
                  f"{CPU_THREADS} BLAS threads",
    }


GEMV_SHAPES = (   # config 1: (name, rows, K, RMSNorm prologue, argmax epilogue)
    ("qkv", 1152, 896, True, False),
    ("gate_up", 9728, 896, True, False),
    ("down", 896, 4864, False, False),
    ("lm_head", 151936, 896, True, True),
)


def gemv_config1() -> dict:
    """Config 1: the q4 GEMV on its own, each shape with enough rotated weight copies to
    exceed 512 MB (past the 256 MB MALL). Bytes per run = codes + (scale, min) pairs."""
    from instantllm_amd import synth
    from instantllm_amd.engine import Gemv
    out = {}
    for name, rows, K, norm, amax in GEMV_SHAPES:
        codes, sb = synth.microbench_q4(1, rows, K)
        x, gamma = synth.microbench_x(1, K)
        nbytes = rows * K // 2 + rows * (K // 64) * 4
        copies = max(2, -(-(512 << 20) // nbytes) + 1)
        g = Gemv(codes, np.ascontiguousarray(sb).view(np.uint32).reshape(rows, K // 64), copies=copies)
        _, _, us = g.run(x[0], gamma if norm else None, iters=max(copies, 20), argmax=amax)
        info = g.info()
        g.close()
        gbs = nbytes / (us * 1e-6) / 1e9
        out[name] = {"rows": rows, "K": K, "bytes": nbytes, "us": round(us, 2), "GBps": round(gbs, 1),
                     "frac": round(gbs / HBM_PEAK_GBS, 4), "copies": copies, "slices": info["slices"]}
    return out


# prefill work of config 4 (M = 512): 2 flops per weight and row over the 24 layers'
# matrices, the lm_head on the last row, and causal attention (QK and PV, 64 dims, 14 heads)
LAYER_PARAMS = 357_826_560
LMH_PARAMS = 136_134_656


def prefill_flops(m: int, layers: int = 24) -> float:
    attn = layers * 14 * 2 * 2 * 64 * (m * (m + 1) / 2)
    return 2.0 * m * LAYER_PARAMS + 2.0 * LMH_PARAMS + attn


def config4(steps: int = 64, single: bool = False) -> dict:
    """Config 4: q8 (symmetric group-64) and f16 models (seed 4): a 512-token prefill on the
    MFMA GEMMs, then `steps` graph-captured greedy decode steps; then the same after a
    4032-token prompt, so the last step attends 4096 positions. With `single` the decode
    steps are launched one by one (for profilers) and timed by HIP events around each."""
    from instantllm_amd import synth, illfile as F
    from instantllm_amd.engine import Engine
    no_eos = (-5, -5)
    out = {}
    for name, fmt in (("q8", F.FMT_Q8), ("f16", F.FMT_F16)):
        e = Engine(synth.cached_model(fmt, 4), max_context=4160, max_pass=16, max_steps=256)
        rng = np.random.default_rng(4)
        prompt = [int(t) for t in rng.integers(0, F.VOCAB, size=512)]
        pre_ms = []
        for _ in range(3):
            e.reset_out_tokens()
            e.set_state(pos=0, n=512, maxsteps=steps + 1, eos=no_eos)
            e.prefill(prompt)
            pre_ms.append(e.last_pass_ms())
        def decode() -> float:
            if single:
                ms = 0.0
                for _ in range(steps):
                    e.decode_step()
                    ms += e.last_pass_ms()
                return ms
            e.capture_steps(steps)
            return e.time_graph(1)

        dec_ms = decode()
        longp = [int(t) for t in rng.integers(0, F.VOCAB, size=4032)]
        e.reset_out_tokens()
        e.set_state(pos=0, n=len(longp), maxsteps=steps + 1, eos=no_eos)
        e.prefill(longp)
        long_ms = decode()
        pos_end = e.get_state()["pos"]
        e.close()
        pm = float(np.median(pre_ms))
        out[name] = {"prefill512_ms": round(pm, 3),
                     "prefill512_tflops": round(prefill_flops(512) / (pm * 1e-3) / 1e12, 1),
                     "decode_us_after_512": round(dec_ms * 1e3 / steps, 1),
                     "decode_us_4032_to_4096": round(long_ms * 1e3 / steps, 1),
                     "last_pos": pos_end}
    return out


def speculative(path: str, n_new: int = 96) -> dict:
    """Speculative generation on the config-2 model (not the headline workload): the learned
    drafter with a table built from the model's own greedy outputs of 8 requests
    (instantllm_amd.ildraft; random scorer weights with the n-gram / self-repetition /
    neighbour features emphasized). `seen`: requests whose outputs the table holds (drafts
    mostly right: an upper end); `unseen`: new requests (drafts mostly wrong: the cost of
    speculating when it does not pay). Tokens equal plain greedy decoding in every run
    (checked); tok/s from the host clock over each whole generate call."""
    import tempfile
    from instantllm_amd import ildraft as DW, illfile as F
    from instantllm_amd.engine import Engine
    e = Engine(path, max_context=1024, max_pass=16, max_steps=n_new + 32)
    rng = np.random.default_rng(11)
    words = ["w%d" % i for i in range(300)]
    def req():
        return [int(t) for t in rng.integers(100, F.VOCAB, 24)], " ".join(rng.choice(words, 6))
    seen = [req() for _ in range(8)]
    unseen = [req() for _ in range(3)]
    recs = [{"prompt": t, "pids": p, "y": e.generate(p, max_new=n_new, chunk=8)} for p, t in seen]
    out = {"n_new": n_new,
           "note": "learned drafter, table from the model's own greedy outputs of 8 requests; seen = requests "
                   "the table holds (drafts mostly right), unseen = new requests; tokens checked equal to greedy (both from a cold prefix cache); "
                   "tok/s from the host clock over whole generate calls"}
    with tempfile.TemporaryDirectory() as td:
        tp = os.path.join(td, "t.bin")
        DW.save(tp, recs, DW.TableSpec(), DW.random_scorer(16, seed=5, emphasis={1: 3.0, 2: 1.5, 17: 2.0, 20: 1.0, 23: 1.5}), {})
        e.load_ildraft(tp)

    def timed(fn):
        fn()   # warm (graph capture)
        t0 = time.perf_counter()
        r = fn()
        return r, time.perf_counter() - t0

    for name, group in (("seen", seen[:3]), ("unseen", unseen)):
        res = {}
        for label, tree, rows in (("greedy", None, 1), ("commit_drafter_chain4", 0, 4), ("learned_chain8", 0, 8),
                                  ("learned_tree16", 15, 16), ("learned_tree16_adaptive", 15, 16),
                                  ("commit_drafter_16_adaptive", 0, 16)):
            toks_n, secs, passes, acc = 0, 0.0, 0, 0
            for p, t in group:
                def greedy():
                    e.truncate_cache(0)   # every run from a cold prefix cache
                    return e.generate(p, max_new=n_new, chunk=8)
                g = greedy()
                if label == "greedy":
                    (_, dt) = timed(greedy)
                    toks_n += len(g); secs += dt
                    continue
                def run():
                    e.truncate_cache(0)
                    if label.startswith("learned"):
                        e.set_learned(True, 8, tree)
                        e.set_draft_context(p, t, None)
                    return e.generate_spec(p, n_new, rows=rows, chunk=4, adaptive=label.endswith("adaptive"))
                (toks, np_, na), dt = timed(run)
                if toks != g:
                    raise RuntimeError(f"speculative tokens differ from greedy ({label}, {name})")
                toks_n += len(toks); secs += dt; passes += np_; acc += na
            res[label] = {"tok_s": round(toks_n / secs, 1)}
            if label != "greedy":
                res[label]["accepted_per_pass"] = round(acc / max(passes, 1), 2)
        out[name] = res
    e.close()
    return out


def speculative_single(path: str, n_new: int = 96) -> dict:
    """The learned drafter's passes of `speculative` launched one at a time (every verify
    pass and every drafting kernel a dispatch of its own), for kernel traces: the profiler
    does not survive a hipGraph launch here. Tree (15 drafts) and chain (7) requests."""
    import tempfile
    from instantllm_amd import ildraft as DW, illfile as F
    from instantllm_amd.engine import Engine
    e = Engine(path, max_context=1024, max_pass=16, max_steps=n_new + 32)
    rng = np.random.default_rng(11)
    words = ["w%d" % i for i in range(300)]
    seen = [([int(t) for t in rng.integers(100, F.VOCAB, 24)], " ".join(rng.choice(words, 6))) for _ in range(8)]
    recs = [{"prompt": t, "pids": p, "y": e.generate(p, max_new=n_new, chunk=8)} for p, t in seen]
    with tempfile.TemporaryDirectory() as td:
        tp = os.path.join(td, "t.bin")
        DW.save(tp, recs, DW.TableSpec(), DW.random_scorer(16, seed=5, emphasis={1: 3.0, 2: 1.5, 17: 2.0, 20: 1.0, 23: 1.5}), {})
        e.load_ildraft(tp)
    out = {}
    for label, tree in (("learned_tree16", 15), ("learned_chain8", 0)):
        passes = acc = 0
        for p, t in seen[:3]:
            e.truncate_cache(0)
            e.set_learned(True, 8, tree)
            e.set_draft_context(p, t, None)
            e.reset_out_tokens()
            e.set_prompt(p)
            e.set_state(pos=0, n=len(p), maxsteps=n_new, tspec=tree + 1 if tree else 8, learned=1)
            e.prefill(p)
            for _ in range(n_new):
                if e.get_state()["done"]:
                    break
                e.spec_pass()
            st = e.get_state()
            passes += st["passes"]
            acc += st["accepted"]
        out[label] = {"passes": passes, "accepted": acc}
    e.close()
    return out


# Trace slots of the pass kernel's per-workgroup timeline (ill_trace_enable): per layer
# ILL_TRL = 16 slots, then the lm_head / commit tail. The 1-row roles mark these stages:
TRACE_TRL, TRACE_TAIL = 16, 16 * 30
ATT_STAGES = (("input coded", 1), ("QKV tiles", 3), ("QKV epilogue", 4), ("attention (wave 0)", 6),
              ("slot states", 14), ("combine", 7), ("O issued", 10))
GUD_STAGES = (("input coded", 1), ("gate/up tile", 3), ("SiLU barrier", 4), ("down coding", 5),
              ("down issued", 10))


def layer_trace(e, prompt: list[int], steps: int) -> dict:
    """The benchmarked configuration with the in-kernel trace on: `steps` decode steps after
    the prefix, captured in one hipGraph and replayed; the trace holds the last step's
    per-workgroup timestamps (100 MHz device clock). Per layer (medians over layers 2-21,
    us from the attention workgroup 0's layer start): the stages of the ATT (workgroups
    0-13) and GUD (16-91) roles; the tail (final norm, lm_head, commit) from the last
    layer's start; the kernel's edges (workgroups entering, the pass header loaded, the
    first layer's start, the commit, workgroups leaving) from the first entry; the step's
    in-kernel span against the graph's per-step time, with and without the trace."""
    no_eos = (-5, -5)

    def replay(trace: bool) -> float:
        e.trace_enable(False)
        if trace:
            e.trace_enable(True)
        e.reset_out_tokens()
        e.set_state(pos=0, n=len(prompt), maxsteps=steps + 64, eos=no_eos)
        e.prefill(prompt)
        e.capture_steps(steps)
        e.sync()
        return e.time_graph(1) * 1e3 / steps

    plain_us = replay(False)
    traced_us = replay(True)
    tr = e.trace_read().astype(np.int64)
    e.trace_enable(False)
    t0 = tr[tr > 0].min()
    rel = np.where(tr > 0, (tr - t0) / 100.0, np.nan)   # us from the step's first mark
    a0 = rel[0, 0::TRACE_TRL][:24]
    layers = range(2, 22)

    def med(wgs, slot):
        v = [rel[w, TRACE_TRL * l + slot] - a0[l] for w in wgs for l in layers]
        return round(float(np.nanmedian(v)), 2)

    att, gud = range(0, 14), range(16, 92)
    tail = {name: round(float(np.nanmedian(rel[:, TRACE_TAIL + k] - a0[23])), 2)
            for name, k in (("final norm coded (median workgroup)", 1), ("lm_head done (median workgroup)", 2))}
    tail["lm_head done (last workgroup)"] = round(float(np.nanmax(rel[:, TRACE_TAIL + 2]) - a0[23]), 2)
    tail["partials seen by the commit"] = round(float(rel[0, TRACE_TAIL + 4] - a0[23]), 2)
    tail["commit done"] = round(float(rel[0, TRACE_TAIL + 5] - a0[23]), 2)
    span = float(np.nanmax(rel))
    entry = rel[:, TRACE_TAIL + 8]
    edges = {"first workgroup entered": 0.0,
             "last workgroup entered": round(float(np.nanmax(entry)), 2),
             "header loaded (median workgroup)": round(float(np.nanmedian(rel[:, TRACE_TAIL + 9])), 2),
             "first layer start (attention workgroup 0)": round(float(a0[0]), 2),
             "commit done": round(float(rel[0, TRACE_TAIL + 5]), 2),
             "workgroup 0 exits": round(float(rel[0, TRACE_TAIL + 10]), 2),
             "last workgroup exits": round(float(np.nanmax(rel[:, TRACE_TAIL + 10])), 2)}
    return {
        "prefix": len(prompt), "steps": steps,
        "graph_us_per_step": round(plain_us, 2), "graph_us_per_step_traced": round(traced_us, 2),
        "in_kernel_span_us_traced": round(span, 2),
        "layer_period_us": round(float((a0[21] - a0[2]) / 19), 3),
        "att_stages_us": {n: med(att, k) for n, k in ATT_STAGES},
        "gud_stages_us": {n: med(gud, k) for n, k in GUD_STAGES},
        "next_layer_att_input_us": round(float(np.nanmedian([a0[l + 1] - a0[l] + rel[0, TRACE_TRL * (l + 1) + 1] - a0[l + 1]
                                                              for l in layers])), 2),
        "tail_from_last_layer_start_us": tail,
        "kernel_edges_us": edges,
    }


def main() -> int:
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=64)
    ap.add_argument("--warmup", type=int, default=8)
    ap.add_argument("--prefix", type=int, default=256)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--cpu-steps", type=int, default=32)
    ap.add_argument("--no-gemv", action="store_true", help="skip the config-1 GEMV microbench")
    ap.add_argument("--no-config4", action="store_true", help="skip the q8 / f16 prefill and decode runs")
    ap.add_argument("--no-spec", action="store_true", help="skip the speculative-decoding runs")
    ap.add_argument("--dispatch", choices=("graph", "single"), default="graph",
                    help="graph: the timed steps are one captured hipGraph (default); single: each "
                         "step is its own launch, timed with HIP events around its kernel, and prompts "
                         "are prefilled through 16-row passes (for profilers that do not follow graph "
                         "launches)")
    ap.add_argument("--spec-single", action="store_true",
                    help="only run the learned drafter's passes one launch at a time (for kernel traces)")
    ap.add_argument("--layer-trace", action="store_true",
                    help="only run the benchmarked configuration with the in-kernel trace on (graph "
                         "replay, no profiler) and print its per-layer breakdown")
    ap.add_argument("--calib-copy-mib", type=int, default=0,
                    help="only run a plain device copy of this many MiB (the reference dispatch "
                         "that scales rocprofv3 FETCH_SIZE / WRITE_SIZE readings) and exit")
    args = ap.parse_args()
    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) != 1:
        print("bench.py: this build runs on one GPU only (the decode step does not shard); "
              "run with --gpus 1", file=sys.stderr)
        return 2
    if args.spec_single:
        from instantllm_amd import synth, illfile as F
        print(json.dumps({"spec_single": speculative_single(synth.cached_model(F.FMT_Q4, 2))}), flush=True)
        return 0
    if args.calib_copy_mib > 0:
        import torch
        n = args.calib_copy_mib << 20
        src = torch.ones(n, dtype=torch.uint8, device="cuda:0")
        dst = torch.empty_like(src)
        for _ in range(3):
            dst.copy_(src)
        torch.cuda.synchronize()
        print(json.dumps({"calib_copy_bytes": n, "dispatches": 4}), flush=True)
        return 0
    from instantllm_amd import illfile as F
    from instantllm_amd.engine import Engine
    from instantllm_amd.synth import random_tree

    path = model_path(F.FMT_Q4, 2)
    rng = np.random.default_rng(2)
    prompt = [int(t) for t in rng.integers(0, F.VOCAB, size=args.prefix)]
    K, W = args.steps, args.warmup
    e = Engine(path, max_context=1024, max_pass=16, max_steps=max(4096, K + W + 16))
    no_eos = (-5, -5)   # the reference's idsbench disables the stop ids (main.swift:165)

    single = args.dispatch == "single"

    def prefill(toks: list[int]) -> None:
        if not single:
            e.prefill(toks)
            return
        for i in range(0, len(toks), 16):   # 16-row passes of the pass kernel
            e.prefill(toks[i:i + 16])

    def run(nsteps: int) -> tuple[float, float, float]:
        e.reset_out_tokens()
        e.set_state(pos=0, n=len(prompt), maxsteps=nsteps + 64, eos=no_eos)
        prefill(prompt)
        e.sync()
        if single:
            ms_dev = 0.0
            t0 = time.perf_counter()
            for _ in range(nsteps):
                e.decode_step()
                ms_dev += e.last_pass_ms()   # HIP events around the step's kernel
            t1 = time.perf_counter()
            return (t1 - t0) * 1e3, ms_dev, e.get_state()["pos"]
        e.capture_steps(nsteps)
        e.sync()
        t0 = time.perf_counter()
        ms_dev = e.time_graph(1)   # HIP events around the graph launch on the engine stream
        t1 = time.perf_counter()
        return (t1 - t0) * 1e3, ms_dev, e.get_state()["pos"]

    if args.layer_trace:
        print(json.dumps({"layer_trace": layer_trace(e, prompt, K)}), flush=True)
        e.close()
        return 0
    if W > 0:
        run(W)
    wall_ms, dev_ms, pos_end = run(K)
    if pos_end != len(prompt) + K:
        raise RuntimeError(f"decode did not advance: pos {pos_end}")
    toks = e.out_tokens()[: K + 1].tolist() if not single else []
    us_tok = dev_ms * 1e3 / K
    L_avg = len(prompt) + (K + 1) / 2.0
    achieved = step_bytes(L_avg) / (us_tok * 1e-6) / 1e9

    # 16-row tree-verify pass (config 3): prefix 512, 15 drafts + root
    vr = np.random.default_rng(3)
    vprompt = [int(t) for t in vr.integers(0, F.VOCAB, size=512)]
    e.reset_out_tokens()
    e.set_state(pos=0, n=512, maxsteps=128, eos=no_eos)
    prefill(vprompt)
    st = e.get_state()
    tree = random_tree(vr, 16, F.VOCAB)
    tree[33] = int(e.out_tokens()[st["step"] - 1])
    verify_us = []
    for _ in range(15):   # single launches: the median of 15 (a pass varies by about 10 us)
        e.set_state(pos=st["pos"], n=16, maxsteps=64, eos=no_eos)
        e.verify_pass(16, tree=tree)
        verify_us.append(e.last_pass_ms() * 1e3)
    # 4-row chain pass (passes of 3-4 rows run on the 16-row instantiation; the reference's
    # default speculative pass has 3 rows) at the same prefix: the last token and three drafts
    chain = [int(tree[33])] + [int(t) for t in vr.integers(0, F.VOCAB, size=3)]
    verify4_us = []
    for _ in range(15):
        e.set_state(pos=st["pos"], n=4, maxsteps=64, eos=no_eos)
        e.verify_pass(4, toks=chain)
        verify4_us.append(e.last_pass_ms() * 1e3)
    e.set_state(pos=st["pos"], n=1, maxsteps=64, eos=no_eos)
    one_us = []
    for _ in range(5):
        e.set_state(pos=st["pos"], n=1, maxsteps=64, eos=no_eos)
        e.decode_step()
        one_us.append(e.last_pass_ms() * 1e3)
    e.close()

    line = {
        "metric": METRIC,
        "value": round(K / (dev_ms * 1e-3), 2),
        "unit": "tok/s",
        "n_gpus": 1,
        "steps": K,
        "warmup": W,
        "ms_per_step": round(dev_ms / K, 5),
        "us_per_token": round(us_tok, 2),
        "wall_ms_per_step": round(wall_ms / K, 5),
        "verify16_us": round(float(np.median(verify_us)), 2),
        "verify4_us": round(float(np.median(verify4_us)), 2),
        "decode1_single_launch_us": round(float(np.median(one_us)), 2),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "int8 MFMA (q4 weights, 16-bit fixed-point activations) + f32",
        "data": "synthetic (seeded random weights and token ids)",
        "config": {"workload": "config 2: q4 1-row greedy decode, Qwen2.5-0.5B shape (24L, d896, 14/2 heads, "
                               "FFN 4864, vocab 151936), prefix KV 256, each step one persistent kernel "
                               + ("in a hipGraph" if not single else "launched on its own (--dispatch single)"),
                   "prefix": len(prompt), "model_seed": 2, "first_tokens": toks[:8]},
        "roofline": {"bound": "hbm", "achieved": round(achieved, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
                     "frac": round(achieved / HBM_PEAK_GBS, 4), "traffic": TRAFFIC_BYTES_PER_STEP,
                     "note": f"bytes(L)={step_bytes(L_avg):.0f} at mean L={L_avg:.1f}; dominant kernel "
                             "ill_pass_kernel<1> (the whole step), duration from HIP events "
                             + ("over the timed graph; " if not single else "around each step's kernel; ")
                             + "traffic = HBM bytes per launch from rocprofv3 FETCH_SIZE/WRITE_SIZE "
                             "(profiles/pass_kernel_q4_decode_config2.md)"},
    }
    line["mfma_counters"] = {"source": "profiles/pass_kernel_q4_decode_config2.md, "
                                       "profiles/layer_by_layer_q8_f16_config4.md", **MFMA_COUNTERS}
    if not args.no_gemv:
        line["gemv_config1"] = gemv_config1()
    if not args.no_config4:
        line["config4"] = config4(single=single)
    if not args.no_spec and not single:
        line["speculative"] = speculative(path)
    if not args.no_cpu:
        line["cpu_baseline"] = cpu_baseline(args.cpu_steps)
    print(json.dumps(line), flush=True)
    return 0


if __name__ == "__main__":
    sys.exit(main())
