// Launch plans and index bounds of the layer-by-layer path: plain constexpr functions of sizes,
// used by the host, by the kernels and, compiled by themselves, by the CPU tests.
#pragma once

#define OP_MAXS 24   // K slices of a split GEMM at most

// K slices of a prompt chunk's residual products (O, down; over 112 rows): `tiles` output tiles,
// `nsteps` k-steps, room for `cap` slices of partials. As many as put about one tile on every CU;
// three where that puts up to two tiles on every CU (86-170 tiles, 769-1536 rows; whole prompts,
// unsplit -> three slices, ms: 770 rows 2.67 -> 2.20 q4, 2.81 -> 2.26 q8, 2.67 -> 2.19 f16; 1152 rows
// 3.00 -> 2.58, 3.16 -> 2.66, 2.96 -> 2.61; 1500 rows 3.30 -> 2.94, 3.45 -> 3.03, 3.26 -> 3.00; at
// 2000 and 3000 rows splitting gained nothing). Never two: a trial build that cut the O projection
// into two slices of 7 k-steps ended in an illegal memory access whose cause was not found.
constexpr int op_slices(int tiles, int nsteps, int cap) {
  int s = 3 * tiles <= 512 ? (256 / tiles > 3 ? 256 / tiles : 3) : 1;
  s = s < nsteps / 4 ? s : nsteps / 4;
  s = s < OP_MAXS ? s : OP_MAXS;
  s = s < cap ? s : cap;
  if (s < 3) return 1;
  const int per = (nsteps + s - 1) / s;
  return (nsteps + per - 1) / per;
}

// 64-position chunks that the attention of a row at pos + dep reads (pos .. the row itself
// included), never past the cache: a finished request may stand at pos = maxctx, and the passes of
// 1 to 16 rows still queued behind it compute, without storing, on positions beyond that.
constexpr int row_chunks(int pos, int dep, int maxctx) {
  const int n = (pos + dep + 64) >> 6;
  return n < maxctx / 64 ? n : maxctx / 64;
}
