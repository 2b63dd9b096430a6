"""Launch plans and index bounds of the layer-by-layer path (instantllm_amd/csrc/ill_plan.h),
compiled with the host compiler and evaluated over their whole range on the CPU."""
from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

CSRC = Path(__file__).resolve().parents[1] / "instantllm_amd" / "csrc"
H, FF, NT = 896, 4864, 7              # hidden size, FFN size, 128-column tiles of the residual
ROWS = range(113, 4097)               # prompt chunks on the ring GEMMs
PART_BYTES = 32 << 20


def evaluate(tmp_path, body: str) -> np.ndarray:
    """The integers that a C++ `main` with this body prints, a row a line."""
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("no host compiler")
    src, exe = tmp_path / "plan.cpp", tmp_path / "plan"
    src.write_text('#include <cstdio>\n#include "ill_plan.h"\nint main() {\n' + body + "\n}\n")
    subprocess.run([cxx, "-std=c++17", "-O1", "-Wall", "-Werror", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout
    return np.array([[int(x) for x in line.split()] for line in out.splitlines()])


def test_part_bytes_is_the_engines():
    text = (CSRC / "ill_engine.hip").read_text()
    assert "#define ILL_OP_PART_BYTES (32u << 20)" in text


@pytest.mark.parametrize("k", [H, FF], ids=["o", "down"])
def test_k_slices_of_prompt_products(tmp_path, k):
    """Every chunk's slices hold all of K, none is empty, the partials fit their buffer, and no
    product is cut in two (O: two slices of 7 k-steps)."""
    nsteps = k // 64
    t = evaluate(tmp_path, f"""
      for (int m = {ROWS.start}; m < {ROWS.stop}; m++) {{
        const int s = op_slices({NT} * ((m + 63) / 64), {nsteps}, {PART_BYTES} / (m * {H} * 4));
        printf("%d %d\\n", m, s);
      }}""")
    m, s = t[:, 0], t[:, 1]
    assert np.array_equal(m, np.arange(ROWS.start, ROWS.stop))
    assert not (s == 2).any(), m[s == 2]
    assert (s >= 1).all() and (s <= 24).all()
    per = -(-nsteps // s)
    assert ((s - 1) * per < nsteps).all() and (s * per >= nsteps).all()
    assert (s * m * H * 4 <= PART_BYTES)[s > 1].all()


def test_attention_chunks_stay_inside_the_cache(tmp_path):
    """Every row of a live pass reads all of its positions; a row of a pass queued behind a request
    that ended at the context's limit reads no chunk past the cache."""
    t = evaluate(tmp_path, """
      for (int ctx = 64; ctx <= 4608; ctx += ctx < 1024 ? 64 : 512)
        for (int pos = 0; pos <= ctx; pos++)
          for (int dep = 0; dep < 16; dep += 5) printf("%d %d %d %d\\n", ctx, pos, dep, row_chunks(pos, dep, ctx));""")
    ctx, pos, dep, n = t.T
    assert (64 * n <= ctx).all()
    live = pos + 16 <= ctx
    assert np.array_equal(n[live], -(-(pos + dep + 1)[live] // 64))
    assert (n >= 1).all()


def test_row_attention_takes_its_chunks_from_the_plan():
    text = (CSRC / "ill_rows.h").read_text()
    assert "nch = row_chunks(pos, dep, c.maxctx);" in text
