// Layer-by-layer ("op") path: one kernel per operation, for any number of rows M.
//
// It serves what the persistent q4 pass kernel does not: the prompt prefill, in chunks of up to
// ILL_OP_MAXM rows, and every pass of q8 and f16 models. Up to ROW_MAXM rows run on the row
// kernels (ill_rows.h); longer chunks on the kernels here: GEMMs streamed through an LDS ring,
// MFMA flash attention, and the residual with the next RMSNorm.
//
// It follows the reference's own encoding (Engine.swift:370-403 encodePrefillLayer2 on
// gemm3_core, Shaders.swift:1911-2054; the 1-row kernels :1199-1364): per layer
//   norm(ln1) -> QKV GEMM (+bias, RoPE, K/V cache write) -> attention -> O GEMM (+x)
//   -> norm(ln2) -> gate/up GEMM (SiLU * up) -> down GEMM (+x),
// then the final norm and the lm_head GEMM with an argmax epilogue on the rows that need
// logits, and the commit.
//
// Arithmetic: activations in f16 (the reference's G3 path keeps fp16 activations too),
// weights dequantized to f16 (q4: s*q + m; q8: s*q; f16: as stored),
// v_mfma_f32_16x16x32_f16 with fp32 accumulation over K in a fixed order, fp32 residual
// stream. Passes of up to 16 rows all run on the row kernels, where a row's arithmetic does not depend
// on the rows beside it: a row decoded alone and inside a 16-row pass give identical bits. A
// prompt chunk's K slices and attention shape follow its number of rows.
//
// Every kernel reads the position and the stop flag from the device State, so a decode
// step recorded in a hipGraph replays correctly.
#pragma once
#include "ill_pass.h"
#include "ill_plan.h"

// Rows of a prompt chunk at most (less where the context is shorter). The GEMMs need many rows
// to fill the chip: whole prompts in chunks of 1280 / 2048 / 4096 rows, ms: 4000 tokens q4 11.7 / 8.7 /
// 7.1, q8 11.7 / 9.2 / 7.4, f16 11.2 / 8.7 / 7.2; 3000 tokens q4 8.3 / 7.0 / 5.6; 2500 tokens q4
// 6.0 / 6.1 / 4.9. The activations of 4096 rows take 90 MB.
#define ILL_OP_MAXM 4096

struct OpMat {
  const uint8_t* w;    // q4 nibbles, q8 int8 or f16 halves, tiled (op_wt_off, op_w4_off)
  const uint16_t* s;   // q4: f16 (scale, min) pairs, q8: f16 scales, tiled (op_st_off); f16: unused
  int N, K, qg;        // qg: q8 group size (32 or 64)
};

// The matrices of the layer-by-layer path are tiled, so that a wave's 16-byte
// loads of one k-step (64 columns) read whole cache lines: 128-row blocks, k-steps, 16-row
// sub-tiles of 16 x 64 weights, inside which 16-byte units are ordered (8-column half e,
// 16-column group kg, row n). Element (r, k) of an N x K matrix of es-byte weights (N a
// multiple of 128, K of 64) lies at byte op_wt_off:
//   ((((r >> 7) * (K / 64) + (k >> 6)) * 8 + ((r & 127) >> 4)) * 64 es
//    + ((e * 4 + kg) * 16 + (r & 15)) * 16 + (k & 7) * es)   with kg = (k & 63) >> 4,
//   e = (k >> 3) & 1 for f16; for q8 a unit holds 16 columns (e = 0, (k & 15) bytes).
// A lane (kg, n) then reads 1 KB contiguous with its wave. q8 scales: [block][k-step]
// [128 rows][64 / qg] (op_st_off). q4: a lane (kg, n)'s 16 columns are two dwords of 8
// nibbles (512 bytes per sub-tile, op_w4_off), column 2 i + j of the 8 in nibble i + 4 j, so
// that (word >> 4 i) & 0x000f000f holds two neighbouring columns; (scale, min) pairs
// [block][k-step][128 rows].
__host__ __device__ inline size_t op_wt_off(int r, int k, int K, int es) {
  const size_t tile = ((size_t)(r >> 7) * (K >> 6) + (k >> 6)) * 8 + ((r & 127) >> 4);
  const int kg = (k & 63) >> 4;
  if (es == 1) return tile * 1024 + (size_t)((kg * 16 + (r & 15)) * 16 + (k & 15));
  const int e = (k >> 3) & 1;
  return tile * 2048 + (size_t)(((e * 4 + kg) * 16 + (r & 15)) * 16 + (k & 7) * 2);
}
__host__ __device__ inline size_t op_st_off(int r, int k, int K, int qg) {
  return (((size_t)(r >> 7) * (K >> 6) + (k >> 6)) * 128 + (r & 127)) * (64 / qg) + ((k & 63) / qg);
}

__host__ __device__ inline size_t op_w4_off(int r, int k, int K) {   // of the dword with column k
  const size_t tile = ((size_t)(r >> 7) * (K >> 6) + (k >> 6)) * 8 + ((r & 127) >> 4);
  return tile * 512 + (size_t)((((k & 63) >> 4) * 16 + (r & 15)) * 8 + ((k >> 3) & 1) * 4);
}

struct OpLayerW {
  OpMat qkv, o, gu, d;
  const float* bqkv;
  const float* ln1;
  const float* ln2;
};

struct OpCtx {
  const OpLayerW* L;
  OpMat emb;             // embedding = tied lm_head
  const float* fnorm;
  IllState* st;
  IllCtl* ctl;
  int32_t* ptoks;        // [M] row tokens (commit writes [0])
  const int32_t* tree;   // [65]
  const float2* rope;
  uint16_t* kc;
  uint16_t* vt;
  float* x;              // [M][896] residual stream
  __half* xn;            // [M][896] normalized activations
  float* q;              // [M][896] queries
  __half* ao;            // [M][896] attention output
  __half* h;             // [M][4864] SiLU(gate) * up
  uint64_t* amax;        // [16][V/128] argmax keys of the lm_head tiles
  float* logits;         // [16][V]
  int maxctx, layers, vocab;
  int kvswz;             // K/V cache layout: 1 swizzled (q8 / f16), 0 rows (q4; ill_common.h)
};

// What the kernels need from the State and the control block, read once at kernel entry
// together with their first operands (a load that gates the others would add a memory round
// trip to every kernel); `done` is checked before the first store.
struct OpHdr {
  int done, pos, mode, wlog;
};
__device__ __forceinline__ OpHdr op_hdr(const OpCtx& c) {
  OpHdr h;
  h.done = gld(&c.st->done);
  h.pos = gld(&c.st->pos);
  h.mode = gld(&c.ctl->mode);
  h.wlog = gld(&c.ctl->write_logits);
  return h;
}

// Row t's position offset from pos (its depth): tree passes read the tree, others are chains.
__device__ __forceinline__ int op_depth(const OpCtx& c, int mode, int t) {
  return mode == ILL_MODE_TREE ? gld(c.tree + ILL_TR_DEPTH + t) : (mode == ILL_MODE_DECODE ? 0 : t);
}

// ---- embedding and RMSNorm -----------------------------------------------------------
template <int FMT>
__device__ __forceinline__ float op_dequant1(const OpMat& m, int r, int k) {
  if constexpr (FMT == 2) {
    const uint32_t x = *(const uint32_t*)(m.w + op_w4_off(r, k, m.K));
    const float q = (float)((x >> (4 * (((k & 7) >> 1) + 4 * (k & 1)))) & 15);
    const uint32_t sm = *((const uint32_t*)m.s + op_st_off(r, k, m.K, 64));
    return h2f(sm & 0xffff) * q + h2f(sm >> 16);
  } else if constexpr (FMT == 1) {
    const float q = (float)(int8_t)m.w[op_wt_off(r, k, m.K, 1)];
    return h2f(m.s[op_st_off(r, k, m.K, m.qg)]) * q;
  } else {
    return h2f(*(const uint16_t*)(m.w + op_wt_off(r, k, m.K, 2)));
  }
}

// xn[t] = f16(x[t] * rsqrt(mean(x^2) + eps) * gamma) for rows row0 .. row0 + M - 1 (one wave
// per row; sum of squares in a fixed order). Output row index t - row0.
__global__ __launch_bounds__(256) void op_norm_kernel(OpCtx c, const float* gamma, int row0, int M) {
  const int done = gld(&c.st->done);
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int t = blockIdx.x * 4 + w;
  if (t >= M) return;
  const float* xr = c.x + (size_t)(row0 + t) * ILL_H;
  float v[14], g[14];
#pragma unroll
  for (int i = 0; i < 14; i++) {
    v[i] = gld(xr + 64 * i + lane);
    g[i] = gld(gamma + 64 * i + lane);
  }
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < 14; i++) ss += v[i] * v[i];
  ss = gsum<64>(ss);
  const float scale = __builtin_amdgcn_rsqf(ss * (1.0f / (float)ILL_H) + ILL_EPS);
  if (done) return;
#pragma unroll
  for (int i = 0; i < 14; i++)
    gst((uint16_t*)(c.xn + (size_t)t * ILL_H + 64 * i + lane), (uint16_t)__half_as_ushort(__float2half(v[i] * scale * g[i])));
}

// The embedding rows of the pass's tokens (Shaders.swift:118-126, :179-190) into x and, from the same registers, layer 0's
// RMSNorm of them into xn, in one launch (one wave per row; the sum of squares in
// op_norm_kernel's order).
template <int FMT>
__global__ __launch_bounds__(256) void op_embed_norm_kernel(OpCtx c, const float* gamma, int M) {
  const int done = gld(&c.st->done);
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int t = blockIdx.x * 4 + w;
  if (t >= M) return;
  const int tok = gld(c.ptoks + t);
  float v[14], g[14];
#pragma unroll
  for (int i = 0; i < 14; i++) {
    v[i] = op_dequant1<FMT>(c.emb, tok, 64 * i + lane);
    g[i] = gld(gamma + 64 * i + lane);
  }
  float* xr = c.x + (size_t)t * ILL_H;
  if (!done) {
#pragma unroll
    for (int i = 0; i < 14; i++) gst(xr + 64 * i + lane, v[i]);
  }
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < 14; i++) ss += v[i] * v[i];
  ss = gsum<64>(ss);
  const float scale = __builtin_amdgcn_rsqf(ss * (1.0f / (float)ILL_H) + ILL_EPS);
  if (done) return;
#pragma unroll
  for (int i = 0; i < 14; i++)
    gst((uint16_t*)(c.xn + (size_t)t * ILL_H + 64 * i + lane), (uint16_t)__half_as_ushort(__float2half(v[i] * scale * g[i])));
}

// ---- GEMM: Y[M][N] = A[M][K] (f16) * W[N][K]^T, fused epilogues ------------------------
enum OpEpi { OP_QKV = 0, OP_RESID = 1, OP_SILU = 2, OP_LMH = 3 };

struct OpGemmArgs {
  OpCtx c;
  const __half* A;   // [M][K]
  OpMat W;
  int M, layer;
  float* resid;      // OP_RESID: [M][896] += Y
  float* part;       // split K: [slices][M][N] fp32 partials
  int ksteps;        // 64-column steps per K slice
  int pos_hint;         // the State's pos as the host expects it (QKV epilogue: rotary rows
                        // are loaded for pos_hint + row with the partials)
};

#define OP_BN 128
#define OP_HLD 72    // LDS row stride (halves) of a gate/up tile's hidden units
#define OP_BK 64

// q8 dequantization, 4 weights at a time: s * (f16)q for the 4 int8 codes of x. Each code
// q becomes the half 1024 + (q + 128) (exponent 0x64 over the byte q ^ 0x80, built with
// v_perm), from which 1152 is subtracted: both exact, so the products equal
// s * (_Float16)(float)q, computed two at a time on packed f16 (v_pk_add_f16, v_pk_mul_f16).
typedef _Float16 op_h2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void op_q8x4(uint32_t x, _Float16 s, _Float16* o) {
  const uint32_t u = x ^ 0x80808080u;
  const op_h2 k = {(_Float16)1152.f, (_Float16)1152.f}, sc = {s, s};
  const op_h2 a = __builtin_bit_cast(op_h2, __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u)) - k;
  const op_h2 b = __builtin_bit_cast(op_h2, __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u)) - k;
  const op_h2 pa = a * sc, pb = b * sc;
  o[0] = pa[0];
  o[1] = pa[1];
  o[2] = pb[0];
  o[3] = pb[1];
}

// q4 dequantization, the 8 weights of a dword: s * q + m. Nibble pairs under the exponent
// byte 0x64 are the halves 1024 + q; 1024 off is exact, then one fused f16 multiply-add.
__device__ __forceinline__ void op_q4x8(uint32_t x, _Float16 s, _Float16 m, _Float16* o) {
  const op_h2 k = {(_Float16)1024.f, (_Float16)1024.f}, sc = {s, s}, mn = {m, m};
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const op_h2 q = __builtin_bit_cast(op_h2, ((x >> (4 * i)) & 0x000f000fu) | 0x64006400u) - k;
    const op_h2 v = __builtin_elementwise_fma(q, sc, mn);
    o[2 * i] = v[0];
    o[2 * i + 1] = v[1];
  }
}

// ---- epilogues ---------------------
// QKV: one rotary block b = columns 32 b .. +31 holds dims d (x0, columns 32 b + i) and
// d + 32 (x1, columns 32 b + 16 + i) of head b / 2 (Convert.swift:236-244); q heads 0-13,
// k 14-15, v 16-17: bias, RoPE at the row's position, then q or the K / V cache slot.
// cs_at / cs: a rotary row already loaded for position cs_at (-1: none), used when it is
// the row's position; bpre: the two bias values already loaded (nullptr: load them).
__device__ __forceinline__ void epi_qkv(const OpCtx& c, const OpHdr& hd, int layer, int m, int b, int i, float x0, float x1,
                                        int cs_at = -1, float2 cs_pre = make_float2(0.f, 0.f), const float* bpre = nullptr) {
  const int head = b >> 1, d = (b & 1) * 16 + i;
  x0 += bpre ? bpre[0] : gld(c.L[layer].bqkv + 32 * b + i);
  x1 += bpre ? bpre[1] : gld(c.L[layer].bqkv + 32 * b + 16 + i);
  const int pos = hd.pos;
  if (head < ILL_NH + ILL_NKV) {
    const int p = pos + op_depth(c, hd.mode, m);
    const float2 cs = p == cs_at ? cs_pre : gld(c.rope + p * 32 + d);
    const float r0 = x0 * cs.x - x1 * cs.y, r1 = x1 * cs.x + x0 * cs.y;
    x0 = r0;
    x1 = r1;
  }
  const int slot = pos + m;
  if (head < ILL_NH) {
    c.q[(size_t)m * ILL_H + head * 64 + d] = x0;
    c.q[(size_t)m * ILL_H + head * 64 + d + 32] = x1;
  } else if (head < ILL_NH + ILL_NKV) {
    uint16_t* kb = c.kc + ((size_t)layer * ILL_NKV + (head - ILL_NH)) * c.maxctx * 64;
    kb[kv_k_off(slot, d, c.kvswz)] = (uint16_t)f2h(x0);
    kb[kv_k_off(slot, d + 32, c.kvswz)] = (uint16_t)f2h(x1);
  } else {
    uint16_t* vb = c.vt + ((size_t)layer * ILL_NKV + (head - ILL_NH - ILL_NKV)) * (c.maxctx / 64) * 4096;
    vb[kv_v_off(slot, d, c.kvswz)] = (uint16_t)f2h_sat(x0);
    vb[kv_v_off(slot, d + 32, c.kvswz)] = (uint16_t)f2h_sat(x1);
  }
}
// gate/up rows in groups of 4: g[2q], g[2q+1], u[2q], u[2q+1] (Convert.swift:134-136)
// SiLU(g) * u, shared by prompts and passes of up to 16 rows. (exp2 of a rounded product and the
// hardware reciprocal instead lose bits of fp32: gate/up of 2000 rows 51.3 us against 55.1, f16.)
__device__ __forceinline__ __half silu_mul(float g, float u) { return __float2half(g / (1.0f + expf(-g)) * u); }
__device__ __forceinline__ void epi_silu(const OpCtx& c, int m, int unit, float g, float u) {
  c.h[(size_t)m * ILL_FF + unit] = silu_mul(g, u);
}

// Epilogue of a 128-column tile (lane (kg, n) of wave w holds rows m0 + 16 i + 4 kg + r,
// columns n0 + 32 w + 16 j + n): fp32 partials of a K slice, or the fused epilogue.
// QKV: cs_base >= 0 gives the rotary rows cs[4 i + r] of rows m0 + 16 i + 4 kg + r at
// position cs_base + row (used when that is the row's position); qbias: the lane's two bias
// values, already loaded (nullptr: loaded here).
template <int BM, int EPI>
__device__ __forceinline__ void op_gemm_epilogue(const OpGemmArgs& a, const OpHdr& hd, const v4f (&acc)[BM / 16][2], int m0,
                                                 int n0, int kz, int w, int kg, int n, uint64_t (&red)[4][16],
                                                 int cs_base = -1, const float2* cs = nullptr, const float* qbias = nullptr,
                                                 uint16_t* hst = nullptr) {
  constexpr int TM = BM / 16;
  if (hd.done) return;
  const OpCtx& c = a.c;
  const int tid = threadIdx.x;
  if (gridDim.z > 1) {   // split K: partials for op_epi_norm_kernel
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int j = 0; j < 2; j++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int m = m0 + 16 * i + 4 * kg + r, col = n0 + 32 * w + 16 * j + n;
          if (m < a.M) a.part[((size_t)kz * a.M + m) * a.W.N + col] = acc[i][j][r];
        }
    return;
  }
  // ---- fused epilogues: lane holds rows 16 i + 4 kg + r, columns n0 + 32 w + 16 j + n
  if constexpr (EPI == OP_RESID) {
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int j = 0; j < 2; j++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int m = m0 + 16 * i + 4 * kg + r, col = n0 + 32 * w + 16 * j + n;
          if (m < a.M) a.resid[(size_t)m * ILL_H + col] += acc[i][j][r];
        }
  } else if constexpr (EPI == OP_SILU) {
    // Lanes n % 4 = 0, 1 hold the gate values of units 2 q, 2 q + 1 and lanes 2, 3 their up
    // values. The quad's halves swap rows (quad_perm 2 3 0 1): lanes 0, 1 then apply rows
    // 4 kg + 0, 1 and lanes 2, 3 rows 4 kg + 2, 3, so that every lane computes two units.
    const bool lo = (n & 3) < 2;
    const int u = (n & 3) - (lo ? 0 : 2);
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int j = 0; j < 2; j++) {
        const int col = n0 + 32 * w + 16 * j + n;
#pragma unroll
        for (int h = 0; h < 2; h++) {
          const float mine = acc[i][j][lo ? h : 2 + h], send = acc[i][j][lo ? 2 + h : h];
          const float got = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(send), 0x4e, 0xf, 0xf, false));
          // into the tile's f16 image in LDS (64 units a row), then stored 16 bytes per lane
          // (2-byte stores from here: 70 us at 2000 rows, f16, when the rest of the kernel made it 66)
          hst[(16 * i + 4 * kg + (lo ? h : 2 + h)) * OP_HLD + ((col - n0) >> 2) * 2 + u] =
              __half_as_ushort(silu_mul(lo ? mine : got, lo ? got : mine));
        }
      }
    lds_barrier();
#pragma unroll
    for (int q = 0; q < BM / 32; q++) {
      const int r = 32 * q + (tid >> 3), e = 8 * (tid & 7);
      if (m0 + r < a.M) gst((gu32x4*)(c.h + (size_t)(m0 + r) * ILL_FF + n0 / 2 + e), *(const gu32x4*)(hst + r * OP_HLD + e));
    }
  } else if constexpr (EPI == OP_QKV) {
    const int b = (n0 + 32 * w) >> 5;
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int m = m0 + 16 * i + 4 * kg + r;
        if (m < a.M) {
          if (cs_base >= 0) epi_qkv(c, hd, a.layer, m, b, n, acc[i][0][r], acc[i][1][r], cs_base + m, cs[4 * i + r], qbias);
          else epi_qkv(c, hd, a.layer, m, b, n, acc[i][0][r], acc[i][1][r], -1, make_float2(0.f, 0.f), qbias);
        }
      }
  } else {   // OP_LMH: logits (optional) and per-tile argmax keys per row (BM == 16)
    const int wlog = hd.wlog;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int m = 4 * kg + r;
      uint64_t k = 0;
#pragma unroll
      for (int j = 0; j < 2; j++) {
        const int col = n0 + 32 * w + 16 * j + n;
        const float v = acc[0][j][r];
        if (wlog && m < a.M) c.logits[(size_t)m * c.vocab + col] = v;
        const uint64_t kk = amax_key(v, col);
        k = kk > k ? kk : k;
      }
      for (int o = 8; o >= 1; o >>= 1) {
        const uint64_t ok = __shfl_xor(k, o, 64);
        k = ok > k ? ok : k;
      }
      if (n == 0) red[w][m] = k;
    }
    __syncthreads();
    if (tid < 16) {
      uint64_t k = red[0][tid];
      for (int ww = 1; ww < 4; ww++) k = red[ww][tid] > k ? red[ww][tid] : k;
      c.amax[(size_t)tid * gridDim.x + blockIdx.x] = k;
    }
  }
}

// Tile of a prefill GEMM workgroup (grid: column tiles x row tiles x K slices). Workgroups
// are dealt to the 8 XCDs round-robin (workgroup id mod 8), and each XCD has its own L2, so
// the tiles are renumbered: the order (K slice, column tile, row tile) is cut into 8
// contiguous runs, run c going to the workgroups on XCD c in dispatch order. The row tiles
// of a weight slab (column tile, K slice) then share one XCD's L2 instead of fetching the
// slab from HBM once per XCD (512-row down projection, f16: 19.3 -> 16.5 us; QKV and O
// 2-7% faster). A permutation of tiles: the results do not change.
struct OpTile {
  int x, y, z;
};
__device__ __forceinline__ OpTile op_tile_xcd() {
  const int nx = gridDim.x, ny = gridDim.y;
  const int T = nx * ny * gridDim.z;
  const int id = blockIdx.x + nx * (blockIdx.y + ny * blockIdx.z);
  const int c = id & 7, k = id >> 3;
  const int u = c * (T >> 3) + min(c, T & 7) + k;   // XCD c holds ceil((T - c) / 8) workgroups
  const int y = u % ny, sl = u / ny;
  return {sl % nx, y, sl / nx};
}

// ---- prompt GEMM and lm_head: operands streamed from memory into an LDS ring ----------------
// The operands go from memory straight into LDS (global_load_lds_dwordx4: lane i of a wave's
// load writes 16 bytes at the instruction's LDS address + 16 i), into a ring of ST stages, so
// that ST - 1 k-steps (64 columns) are in
// flight with no registers or LDS stores spent on them. (Per workgroup at 512 rows: 0.7 us
// to issue the prologue, then 0.3-0.7 us per k-step; the gate/up GEMM, three workgroups per
// CU, is bound by the LDS traffic of its k-steps: 24 KB written and 48 KB read, the four
// waves reading the same A rows.) A stage holds
//   A: BM rows x 64 halves, row by row, the 8 16-byte units of a row permuted (k / 8 at place
//      k / 8 ^ row / 2 % 8): eight lanes of a load take a row's whole 128-byte line, and the 16 lanes
//      of an operand read (16 rows) fall on different banks. (Units ordered (row / 16, k / 8,
//      row % 16) read without conflicts too, but each load gathered 16 bytes of 64 places: gate/up,
//      f16, 66 us against 53 at 2000 rows);
//   B: the k-step's block of the tiled weights (128 rows x 64 columns at op_wt_off, 4 KB q4,
//      8 KB q8, 16 KB f16) as stored: its units are already in that order;
//   q8: the block's scales (128 rows x 64 / qg f16, op_st_off), 256 or 512 bytes.
// q8 and q4 weights are dequantized as they leave LDS. The loads are issued in inline assembly: the
// compiler's own tracking of LDS loads in flight made it wait for all of them before some of the stage's LDS reads (it
// could not tell the stages apart), which serialized the ring. The wait for the stage about
// to be read is explicit: vmcnt counts this wave's own loads, and the barrier after it covers
// the other waves' loads and orders every wave's reads of the stage refilled next before the
// refill. (The compiler's waits for its own loads count only the loads it knows of, so they
// wait at least as long as they need: loads complete in issue order.)
#define OP_LDS(p) ((__attribute__((address_space(3))) void*)(p))
// One wave-wide load into LDS: lane i's `bytes` (16 or 4) at global g go to LDS byte address
// lds + bytes * i (lds: the same for every lane).
__device__ __forceinline__ void op_lds_dma16(const void* g, const void* lds) {
  const uint32_t m = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)OP_LDS(lds));
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(m), "v"(g) : "m0");
}
__device__ __forceinline__ void op_lds_dma4(const void* g, const void* lds) {
  const uint32_t m = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)OP_LDS(lds));
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" ::"s"(m), "v"(g) : "m0");
}
// Stages: 24 KB (f16) / 16.5 KB (q8) each at BM 64, 20 / 12.5 KB at BM 32. Rings of 6 (f16)
// and 8 (q8) stages for the GEMMs of at most one workgroup per CU, and for all of them, were
// slower (512-row prefill 1.96 / 2.24 ms against 1.93 / 2.12 ms; 2.17 / 2.55 ms): issuing the
// longer prologue took 2 us instead of 0.7 and the k-steps were hardly faster. The gate/up
// GEMM (608 workgroups at 512 rows) takes 2 (f16) / 3 (q8) stages, so that three workgroups
// fit per CU and all of them run in one round (f16: 1.90 -> 1.86 ms); its launch bounds keep the
// registers to three workgroups too (q8 at 176 registers: 65 us at 2000 rows, at 157: 54).
#define OP_RING_ST(FMT, EPI) ((EPI) == OP_SILU ? ((FMT) == 0 ? 2 : 3) : ((FMT) == 0 ? 3 : 4))
template <int FMT, int BM>
struct OpRing {                                  // sizes in 16-byte units
  static constexpr int A = BM * 8;
  static constexpr int B = FMT == 0 ? 1024 : (FMT == 1 ? 512 : 256);
  static constexpr int SC = FMT == 0 ? 0 : 32;
  static constexpr int N = A + B + SC;
  static constexpr int LA = A >= 256 ? A / 256 : 1;   // A loads per thread (BM 16: waves 2, 3 repeat 0, 1)
  static constexpr int L = LA + B / 256 + (FMT == 0 ? 0 : 1);   // loads per thread and stage
};

// Thread tid's loads of the k-step at k0 into stage st (rows >= M read row M - 1).
template <int FMT, int BM>
__device__ __forceinline__ void op_ring_load(const OpGemmArgs& a, int m0, int n0, int k0, uint4* st, int tid) {
  using R = OpRing<FMT, BM>;
  const int K = a.W.K, wb = tid & ~63;   // wave's first unit of each 256-unit run
#pragma unroll
  for (int u = 0; u < R::LA; u++) {
    // unit p (BM 16: 128 units, which waves 2, 3 load again into the same bytes, so that every
    // wave issues the same loads)
    const int p = (256 * u + tid) & (R::A - 1);
    const int row = min(m0 + (p >> 3), a.M - 1);
    op_lds_dma16(a.A + (size_t)row * K + k0 + 8 * ((p ^ (p >> 4)) & 7), st + ((256 * u + wb) & (R::A - 1)));
  }
  const uint4* blk = (const uint4*)(a.W.w + (FMT == 2 ? op_w4_off(n0, k0, K) : op_wt_off(n0, k0, K, FMT == 0 ? 2 : 1)));
#pragma unroll
  for (int u = 0; u < R::B / 256; u++)
    op_lds_dma16(blk + 256 * u + tid, st + R::A + 256 * u + wb);
  if constexpr (FMT != 0) {   // 64 dwords per wave: all of them (q8, qg 64), or half (q4; q8, qg 32: waves 0, 2 the first)
    const int off = FMT == 2 || a.W.qg == 32 ? ((tid >> 6) & 1) * 64 : 0;
    const uint32_t* sc = FMT == 2 ? (const uint32_t*)a.W.s + op_st_off(n0, k0, K, 64) : (const uint32_t*)(a.W.s + op_st_off(n0, k0, K, a.W.qg));
    op_lds_dma4(sc + off + (tid & 63), (uint32_t*)(st + R::A + R::B) + off);
  }
}

// The A operand of half ks of the k-step in stage st: rows 16 i + n.
__device__ __forceinline__ v8h op_ring_a(const uint4* st, int i, int ks, int kg, int n) {
  return u4_to_v8h(st[(16 * i + n) * 8 + ((4 * ks + kg) ^ (n >> 1))]);
}
// The B operand of half ks of the k-step in stage st: 16-row sub-tile c16 of the weight block.
template <int FMT, int BM>
__device__ __forceinline__ v8h op_ring_b(const uint4* st, int c16, int ks, int kg, int n, int qg) {
  using R = OpRing<FMT, BM>;
  if constexpr (FMT == 0) {
    return u4_to_v8h(st[R::A + c16 * 128 + ((kg & 1) * 4 + 2 * ks + (kg >> 1)) * 16 + n]);
  } else {
    v8h v;
    _Float16 o[8];
    if constexpr (FMT == 2) {
      const uint32_t x = ((const uint32_t*)(st + R::A + c16 * 32))[((2 * ks + (kg >> 1)) * 16 + n) * 2 + (kg & 1)];
      const uint32_t sm = ((const uint32_t*)(st + R::A + R::B))[16 * c16 + n];
      op_q4x8(x, (_Float16)h2f(sm & 0xffff), (_Float16)h2f(sm >> 16), o);
    } else {
      const uint2 q = ((const uint2*)(st + R::A + c16 * 64 + (2 * ks + (kg >> 1)) * 16 + n))[kg & 1];
      const uint16_t* sc = (const uint16_t*)(st + R::A + R::B);
      const _Float16 s = (_Float16)h2f(sc[(16 * c16 + n) * (64 / qg) + (qg == 32 ? ks : 0)]);
      op_q8x4(q.x, s, o);
      op_q8x4(q.y, s, o + 4);
    }
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = o[i];
    return v;
  }
}
// The k-step in stage st: lane (kg, n) of wave w, rows 16 i + n, columns 32 w + 16 j + n.
template <int FMT, int BM>
__device__ __forceinline__ void op_ring_mma(const uint4* st, int w, int kg, int n, int qg, v4f (&acc)[BM / 16][2]) {
#pragma unroll
  for (int ks = 0; ks < 2; ks++) {
    v8h bf[2];
#pragma unroll
    for (int j = 0; j < 2; j++) bf[j] = op_ring_b<FMT, BM>(st, 2 * w + j, ks, kg, n, qg);
#pragma unroll
    for (int i = 0; i < BM / 16; i++) {
      const v8h af = op_ring_a(st, i, ks, kg, n);
#pragma unroll
      for (int j = 0; j < 2; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af, bf[j], acc[i][j], 0, 0, 0);
    }
  }
}

// Wait until at most `later` stages of this wave's loads are in flight (a constant once the
// callers' loops are unrolled), then the workgroup barrier.
template <int N>
__device__ __forceinline__ void op_vm_barrier() {
  static_assert(N >= 0 && N < 64, "vmcnt field");
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_waitcnt lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}
template <int L>
__device__ __forceinline__ void op_ring_wait(int later) {
  switch (later) {
    case 0: op_vm_barrier<0>(); break;
    case 1: op_vm_barrier<L>(); break;
    default: op_vm_barrier<2 * L>(); break;
  }
}

// Grid: column tiles x row tiles x K slices (4 waves; wave w owns columns 32 w .. + 31 of
// the 128-column tile and all BM rows).
template <int FMT, int BM, int EPI, int ST>
__global__ __launch_bounds__(256, EPI == OP_SILU ? 3 : 2) void op_gemm_ring_kernel(OpGemmArgs a) {
  static_assert(ST >= 2 && ST <= 4 && BM >= 16 && BM <= 64 && (EPI != OP_LMH || BM == 16), "ring GEMM shape");
  using R = OpRing<FMT, BM>;
  const OpHdr hd = op_hdr(a.c);
#define OP_RING_ARR(i) __shared__ __attribute__((aligned(16))) uint4 r##i[ST > i ? R::N : 1];
  OP_RING_ARR(0) OP_RING_ARR(1) OP_RING_ARR(2) OP_RING_ARR(3)
#undef OP_RING_ARR
  __shared__ uint64_t red[4][16];   // (the argmax epilogue only)
  auto ring = [&](int d) -> uint4* { return d == 0 ? r0 : d == 1 ? r1 : d == 2 ? r2 : r3; };
  constexpr int TM = BM / 16;
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
  const int kg = lane >> 4, n = lane & 15;
  // (tiles renumbered per XCD for the 32- and 64-row prompt tiles but gate/up, which was no faster
  // that way; the argmax epilogue indexes by blockIdx.x)
  const OpTile tl = EPI != OP_SILU && BM > 16 ? op_tile_xcd() : OpTile{(int)blockIdx.x, (int)blockIdx.y, (int)blockIdx.z};
  const int n0 = tl.x * OP_BN, m0 = tl.y * BM;
  const int K = a.W.K, qg = a.W.qg;
  const int kb = tl.z * a.ksteps * OP_BK;
  const int ns = (min(K, kb + a.ksteps * OP_BK) - kb) / OP_BK;
  v4f acc[TM][2];
#pragma unroll
  for (int i = 0; i < TM; i++) {
    acc[i][0] = (v4f){0.f, 0.f, 0.f, 0.f};
    acc[i][1] = (v4f){0.f, 0.f, 0.f, 0.f};
  }
  // QKV: the epilogue's bias values and rotary rows (at the expected positions pos_hint +
  // row), loaded while the k-steps stream (loaded in the epilogue they cost a memory round
  // trip each, about 4 us per workgroup)
  float2 qcs[EPI == OP_QKV ? TM * 4 : 1];
  float qbias[2];
  if constexpr (EPI == OP_QKV) {
    const int b = (n0 + 32 * w) >> 5;
    const float* bq = a.c.L[a.layer].bqkv + 32 * b + n;
    qbias[0] = gld(bq);
    qbias[1] = gld(bq + 16);
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int r = 0; r < 4; r++)
        qcs[4 * i + r] = gld(a.c.rope + (size_t)min(a.pos_hint + m0 + 16 * i + 4 * kg + r, a.c.maxctx - 1) * 32 + (b & 1) * 16 + n);
  }
  // steps past the slice reload its last one, so that every stage issues the same loads
#pragma unroll
  for (int d = 0; d < ST - 1; d++) op_ring_load<FMT, BM>(a, m0, n0, kb + min(d, ns - 1) * OP_BK, ring(d), tid);
  int s0 = 0;
  for (; s0 + ST <= ns; s0 += ST) {
#pragma unroll
    for (int d = 0; d < ST; d++) {
      op_ring_wait<R::L>(ST - 2);
      op_ring_load<FMT, BM>(a, m0, n0, kb + min(s0 + d + ST - 1, ns - 1) * OP_BK, ring((d + ST - 1) % ST), tid);
      op_ring_mma<FMT, BM>(ring(d), w, kg, n, qg, acc);
    }
  }
#pragma unroll
  for (int d = 0; d < ST - 1; d++)
    if (s0 + d < ns) {
      op_ring_wait<R::L>(ST - 2 - d);
      op_ring_mma<FMT, BM>(ring(d), w, kg, n, qg, acc);
    }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // no LDS load outlives the workgroup
  if constexpr (EPI == OP_QKV) op_gemm_epilogue<BM, EPI>(a, hd, acc, m0, n0, tl.z, w, kg, n, red, a.pos_hint, qcs, qbias);
  else {
    if (EPI == OP_SILU) lds_barrier();   // the ring's stages become the epilogue's tile
    static_assert(EPI != OP_SILU || R::N * 16 >= BM * OP_HLD * 2, "a stage holds the tile");
    op_gemm_epilogue<BM, EPI>(a, hd, acc, m0, n0, tl.z, w, kg, n, red, -1, nullptr, nullptr, (uint16_t*)r0);
  }
}

// Residual split-K reduction of a prompt chunk fused with the RMSNorm that reads the updated
// residual: one workgroup per row m, one thread per column. x[m] += the slices' partials (added in
// slice order), xn[m] = f16(x * rsqrt(mean(x^2) + eps) * gamma), the sum of squares taken per wave
// and the 14 wave sums added in order.
__global__ __launch_bounds__(ILL_H) void op_epi_norm_kernel(OpGemmArgs a, int S, const float* gamma) {
  __shared__ float red[ILL_H / 64];
  const OpHdr hd = op_hdr(a.c);
  const int m = blockIdx.x, j = threadIdx.x, w = j >> 6, lane = j & 63;
  float pz[OP_MAXS];
#pragma unroll
  for (int z = 0; z < OP_MAXS; z++) pz[z] = z < S ? gld(a.part + ((size_t)z * a.M + m) * ILL_H + j) : 0.f;
  float* r = a.resid + (size_t)m * ILL_H + j;
  const float g = gld(gamma + j);
  float y = pz[0];
#pragma unroll
  for (int z = 1; z < OP_MAXS; z++)
    if (z < S) y += pz[z];
  const float v = gld(r) + y;
  if (!hd.done) gst(r, v);
  const float ss = gsum<64>(v * v);
  if (lane == 0) red[w] = ss;
  __syncthreads();
  float tot = 0.f;
#pragma unroll
  for (int i = 0; i < ILL_H / 64; i++) tot += red[i];
  const float scale = __builtin_amdgcn_rsqf(tot * (1.0f / (float)ILL_H) + ILL_EPS);
  if (hd.done) return;
  gst((uint16_t*)(a.c.xn + (size_t)m * ILL_H + j), (uint16_t)__half_as_ushort(__float2half(v * scale * g)));
}

// (m, l, o) of n states combined against their maximum, in index order; states with
// m = -inf (no positions) add nothing, and if all are empty the result is empty too.
template <int N>
__device__ __forceinline__ void att_combine(const float* m, const float* l, const float* o, float& mo, float& lo, float& oo) {
  float mm = m[0];
#pragma unroll
  for (int i = 1; i < N; i++) mm = fmaxf(mm, m[i]);
  float sum = 0.f, acc = 0.f;
  if (mm != -INFINITY) {
#pragma unroll
    for (int i = 0; i < N; i++) {
      const float e = att_exp(m[i] - mm);
      sum = sum + l[i] * e;
      acc = acc + o[i] * e;
    }
  }
  mo = mm;
  lo = sum;
  oo = acc;
}

#define OP_ATTN_UP 14.0f   // log2 of the largest probability (of its share of f16's range)
// ---- attention of prompt chunks of more than 16 rows: MFMA flash attention ----------------
// A wave evaluates 16 rows of one query head against 64-position chunks of the cache (this
// chunk's QKV kernel has written its own keys and values): row t < M sits at position pos + t and
// attends to positions 0 .. pos + t. Scores are K rows x rows of q and outputs V dims x rows
// (v_mfma_f32_16x16x32_f16), so the softmax statistics of row n are lane n's, and the keys of an
// MFMA block are dealt out (block b, row 4 kg + r: key 32 (b / 2) + 8 kg + 4 (b % 2) + r) such
// that the probabilities a lane holds are the next product's operand as they stand: no pass
// through LDS, no reduction across the 16 lanes of a row. q and P are split into f16 high and
// low parts. The sums of the exponentials stay per lane until the end, and the value products
// accumulate onto the output. The next chunk streams in meanwhile. The kernel is bound by the vector
// instructions per score.
// GRP: a workgroup per (16 rows, four or three heads of a KV group), SPL waves per head taking turns
// at the chunks; SPL chunks' keys and values at a time go from memory straight into LDS once for
// the heads (16 KB each, two buffers: the next ones stream in meanwhile). For few blocks (GRP
// false): SPL waves per (16 rows, query head), chunk c to wave c % SPL, their states combined in
// wave order. 2000 rows from position 0: 61 us per layer (q4 79) with scores as rows x keys and P
// turned through LDS, every head reading K and V itself; 40 (101) with the layout above, 44 (45)
// with chunks shared through LDS by seven heads, 37 (39) with two waves per head and the lazy
// maximum, 29 (30) with the heads on two workgroups, so that the causal load evens out; 30.5 since the
// probabilities fill f16's range.
template <bool SWZ, bool GRP, int SPL>   // SWZ: the K/V cache layout (ill_common.h): swizzled for q8 / f16, rows for q4
__global__ __launch_bounds__(64 * SPL * (GRP ? 4 : 1), GRP ? 1 : 2) void op_attn_rows_kernel(OpCtx c, int layer, int M, int blk0) {
  const OpHdr hd = op_hdr(c);
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, kg = lane >> 4, n = lane & 15;
  // GRP: 4 workgroups per block, (KV group, its first four or last three heads), in descending
  // order of the blocks' chunks; the second 256 (a CU's second workgroup) in ascending order
  int id = blockIdx.x;
  if (GRP && (id >> 8) == 1) id = min(511, (int)gridDim.x - 1) - (id - 256);
  const int t0 = 16 * (blk0 + (GRP ? ((int)gridDim.x >> 2) - 1 - (id >> 2) : id));
  const int hw = GRP ? w & 3 : 0;
  const int g = GRP ? (id >> 1) & 1 : (int)blockIdx.y / 7, h = GRP ? 7 * g + 4 * (id & 1) + min(hw, 2 + (~id & 1)) : (int)blockIdx.y;
  const bool live = !GRP || !(id & 1) || hw < 3;   // (the last three heads' fourth wave only loads)
  const int sp = GRP ? w >> 2 : w;   // this wave's chunks: sp, sp + SPL, ..
  const int t = min(t0 + n, M - 1);   // (rows past the last repeat it and are not stored)
  float4 qf[2][2];
#pragma unroll
  for (int ks = 0; ks < 2; ks++)
#pragma unroll
    for (int i = 0; i < 2; i++) qf[ks][i] = gld((const float4*)(c.q + (size_t)t * ILL_H + h * 64 + 32 * ks + 8 * kg) + i);
  const uint16_t* kb = c.kc + ((size_t)layer * ILL_NKV + g) * c.maxctx * 64;
  const uint16_t* vb = c.vt + ((size_t)layer * ILL_NKV + g) * c.maxctx * 64;
  struct Frag {
    uint4 k[4][2], v[4][2];
  };
  auto fetch = [&](int ch, Frag& f) {
#pragma unroll
    for (int b = 0; b < 4; b++)
#pragma unroll
      for (int ks = 0; ks < 2; ks++)
        f.k[b][ks] = gld((const uint4*)(kb + kv_k_off(64 * ch + 32 * (b >> 1) + 8 * (n >> 2) + 4 * (b & 1) + (n & 3), 32 * ks + 8 * kg, SWZ)));
#pragma unroll
    for (int nb = 0; nb < 4; nb++)
#pragma unroll
      for (int s = 0; s < 2; s++) f.v[nb][s] = gld((const uint4*)(vb + kv_v_off(64 * ch + 32 * s + 8 * kg, 16 * nb + n, SWZ)));
  };
  const int pos = hd.pos;
  const int L = pos + t + 1;
  const int nch = (pos + min(t0 + 16, M) + 63) >> 6;   // of the block's last row
  const int full = (pos + t0 + 1) >> 6;                // chunks whole for every row
  auto over_kg = [](float v, auto op) {   // over the lanes of the same row
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_int(v), __float_as_int(v), false, false);
    v = op(__int_as_float((int)a[0]), __int_as_float((int)a[1]));
    const auto q = __builtin_amdgcn_permlane32_swap(__float_as_int(v), __float_as_int(v), false, false);
    return op(__int_as_float((int)q[0]), __int_as_float((int)q[1]));
  };
  // q * log2(e) as f16 pairs (of the product before its rounding to fp32), scaled by the power of two
  // that brings the row's largest dim to f16's range; scores * qback are exponents of 2 (row_attn_kernel)
  constexpr float LG = 1.4426950408889634f, LGL = (float)(1.4426950408889634 - (double)LG);
  v8h qh[2], ql[2];
  float v[2][8], qm = 0.f;
#pragma unroll
  for (int ks = 0; ks < 2; ks++) {
    const float x[8] = {qf[ks][0].x, qf[ks][0].y, qf[ks][0].z, qf[ks][0].w, qf[ks][1].x, qf[ks][1].y, qf[ks][1].z, qf[ks][1].w};
#pragma unroll
    for (int i = 0; i < 8; i++) {
      v[ks][i] = x[i];
      qm = fmaxf(qm, fabsf(x[i]));
    }
  }
  const int qe = max(__builtin_amdgcn_frexp_expf(over_kg(qm, OpMaxF{})), -100);
  const float qup = __builtin_ldexpf(1.f, 15 - qe), qback = __builtin_ldexpf(0.125f, qe - 15);
#pragma unroll
  for (int ks = 0; ks < 2; ks++)
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const float y = v[ks][i] * qup, x = y * LG;
      const _Float16 hi = (_Float16)x;
      qh[ks][i] = hi;
      ql[ks][i] = (_Float16)((x - (float)hi) + fmaf(y, LGL, fmaf(y, LG, -x)));
    }
  // The exponents' reference Mx of a row follows its maximum lazily, OP_ATTN_UP below it: the first
  // chunk sets it, and only when a score exceeds the row's by more than 1 is it moved up and
  // everything summed so far rescaled. Probabilities then reach 2^14 to 2^15, so that their f16
  // pairs hold 24 bits down to 2^-15 of the largest. (With the reference at the maximum and moved at
  // 8, chunks far below it lost half of their bits to f16's subnormals.) The score products start
  // from 0 and the reference is subtracted: started from -Mx the exponents' error is up to 1.8
  // times as large. Both together cost 28.0 -> 30.5 us per layer at 2000 rows.
  float Mx = 0.f, Ls = 0.f;   // Ls: this lane's keys only
  bool first = true;
  v4f O[4];
#pragma unroll
  for (int nb = 0; nb < 4; nb++) O[nb] = (v4f){0.f, 0.f, 0.f, 0.f};
  auto eval = [&](int ch, const Frag& f) {
    v4f sc[4];
#pragma unroll
    for (int b = 0; b < 4; b++) {
      v4f d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 2; ks++) {
        d = __builtin_amdgcn_mfma_f32_16x16x32_f16(u4_to_v8h(f.k[b][ks]), qh[ks], d, 0, 0, 0);
        d = __builtin_amdgcn_mfma_f32_16x16x32_f16(u4_to_v8h(f.k[b][ks]), ql[ks], d, 0, 0, 0);
      }
      sc[b] = d;
    }
    if (ch >= full) {   // (wave-uniform) positions past a row
#pragma unroll
      for (int b = 0; b < 4; b++)
#pragma unroll
        for (int r = 0; r < 4; r++)
          if (64 * ch + 32 * (b >> 1) + 8 * kg + 4 * (b & 1) + r >= L) sc[b][r] = -INFINITY;
    }
    float mc = sc[0][0];
#pragma unroll
    for (int b = 0; b < 4; b++)
#pragma unroll
      for (int r = 0; r < 4; r++) mc = fmaxf(mc, sc[b][r]);
    mc *= qback;
    if (first || __any(mc > Mx + (OP_ATTN_UP + 1.f))) {   // (wave-uniform)
      mc = over_kg(mc, OpMaxF{});
      // (a row with no position in its first chunk stays at 0)
      const float mn = first ? (mc == -INFINITY ? 0.f : mc - OP_ATTN_UP) : fmaxf(mc - OP_ATTN_UP, Mx);
      // (nothing is summed before the first chunk, whose maximum may be far below 0: 0 * 2^-mn would be NaN)
      const float sa = first ? 1.f : __builtin_amdgcn_exp2f(Mx - mn);
      first = false;
      Mx = mn;
      Ls *= sa;
#pragma unroll
      for (int nb = 0; nb < 4; nb++) O[nb] *= sa;
    }
    v8h ph[2], pl[2];
#pragma unroll
    for (int b = 0; b < 4; b++)
#pragma unroll
      for (int r = 0; r < 4; r += 2) {
        const float p0 = __builtin_amdgcn_exp2f(fmaf(sc[b][r], qback, -Mx)), p1 = __builtin_amdgcn_exp2f(fmaf(sc[b][r + 1], qback, -Mx));
        Ls += p0;
        Ls += p1;
        const _Float16 h0 = (_Float16)p0, h1 = (_Float16)p1;
        ph[b >> 1][4 * (b & 1) + r] = h0;
        ph[b >> 1][4 * (b & 1) + r + 1] = h1;
        pl[b >> 1][4 * (b & 1) + r] = (_Float16)fmaf((float)h0, -1.f, p0);
        pl[b >> 1][4 * (b & 1) + r + 1] = (_Float16)fmaf((float)h1, -1.f, p1);
      }
#pragma unroll
    for (int nb = 0; nb < 4; nb++)
#pragma unroll
      for (int s = 0; s < 2; s++) {
        O[nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(u4_to_v8h(f.v[nb][s]), ph[s], O[nb], 0, 0, 0);
        O[nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(u4_to_v8h(f.v[nb][s]), pl[s], O[nb], 0, 0, 0);
      }
  };
  __shared__ __attribute__((aligned(16))) uint4 kv[GRP ? 2 : 1][GRP ? SPL * 1024 : 1];
  if constexpr (GRP) {
    // 16-byte units of the chunk as stored (K 0 .. 511, V 512 .. 1023), except that the rows layout's
    // 8 units per key or dim are permuted among themselves, so that the eight lanes that LDS
    // serves at once (fragment reads: keys 0-3 and 8-11, or eight dims) fall on different banks
    auto kswz = [](int key) { return SWZ ? 0 : (key & 3) | ((key >> 1) & 4); };
    auto load = [&](int it, int buf) {   // (chunks past the last repeat it)
      for (int i = w; i < 16 * SPL; i += 4 * SPL) {
        const int u = 64 * (i & 7) + lane, ch = min(SPL * it + (i >> 4), nch - 1);
        const bool k = (i & 15) < 8;
        const int src = SWZ ? u : (u & ~7) | ((u & 7) ^ (k ? kswz(u >> 3) : (u >> 3) & 7));
        op_lds_dma16((const uint4*)((k ? kb : vb) + (size_t)4096 * ch) + src, &kv[buf][64 * i]);
      }
    };
    load(0, 0);
    for (int it = 0; SPL * it < nch; it++) {
      op_vm_barrier<0>();   // these chunks are in LDS, and every wave is done with the buffer filled next
      if (SPL * (it + 1) < nch) load(it + 1, (it + 1) & 1);
      const int ch = SPL * it + sp;
      if (ch >= nch || !live) continue;   // (ch: the last turn)
      Frag f;
      const uint4* b0 = kv[it & 1] + 1024 * sp;
#pragma unroll
      for (int b = 0; b < 4; b++)
#pragma unroll
        for (int ks = 0; ks < 2; ks++) {
          const int key = 32 * (b >> 1) + 8 * (n >> 2) + 4 * (b & 1) + (n & 3), dg = 4 * ks + kg;
          f.k[b][ks] = b0[SWZ ? dg * 64 + key : key * 8 + (dg ^ kswz(key))];
        }
#pragma unroll
      for (int nb = 0; nb < 4; nb++)
#pragma unroll
        for (int s = 0; s < 2; s++) {
          const int dim = 16 * nb + n, pg = 4 * s + kg;
          f.v[nb][s] = b0[512 + (SWZ ? pg * 64 + dim : dim * 8 + (pg ^ (dim & 7)))];
        }
      eval(ch, f);
    }
  } else if (sp < nch) {
    const int c0 = sp;
    Frag f0, f1;
    fetch(c0, f0);
    for (int ch = c0;; ch += 2 * SPL) {   // two chunks per turn: the buffers swap without copies
      // (past the last chunk the fetch repeats it, so the loads in flight never depend on a branch)
      fetch(min(ch + SPL, nch - 1), f1);
      __builtin_amdgcn_sched_barrier(0);
      eval(ch, f0);
      if (ch + SPL >= nch) break;
      fetch(min(ch + 2 * SPL, nch - 1), f0);
      __builtin_amdgcn_sched_barrier(0);
      eval(ch + SPL, f1);
      if (ch + 2 * SPL >= nch) break;
    }
  }
  Ls = over_kg(Ls, OpAddF{});
  if (Ls == 0.f) Mx = -INFINITY;   // a row with no position in this wave's chunks
  if constexpr (GRP) {
    static_assert(SPL == 1 || SPL == 2, "states of two waves per head");
    if constexpr (SPL == 2) {   // the two waves' states, in LDS over the chunks
      float* st = (float*)kv + hw * 18 * 64;
      lds_barrier();
      if (sp == 1) {
        st[lane] = Mx;
        st[64 + lane] = Ls;
#pragma unroll
        for (int nb = 0; nb < 4; nb++) *(v4f*)&st[128 + 256 * nb + 4 * lane] = O[nb];
      }
      lds_barrier();
      if (sp == 1) return;
      const float m1 = st[lane], mm = fmaxf(Mx, m1);
      const float e0 = __builtin_amdgcn_exp2f(Mx - mm), e1 = __builtin_amdgcn_exp2f(m1 - mm);
      Ls = Ls * e0 + st[64 + lane] * e1;
#pragma unroll
      for (int nb = 0; nb < 4; nb++) O[nb] = O[nb] * e0 + *(const v4f*)&st[128 + 256 * nb + 4 * lane] * e1;
    }
    if (hd.done || !live || t0 + n >= M) return;
#pragma unroll
    for (int nb = 0; nb < 4; nb++) {
      uint2 y;
      y.x = f2h(O[nb][0] / Ls) | (f2h(O[nb][1] / Ls) << 16);
      y.y = f2h(O[nb][2] / Ls) | (f2h(O[nb][3] / Ls) << 16);
      gst((gu32x2*)(c.ao + (size_t)t * ILL_H + h * 64 + 16 * nb + 4 * kg), (gu32x2){y.x, y.y});
    }
  } else {
    __shared__ float sm_[SPL][16], sl_[SPL][16];
    __shared__ __attribute__((aligned(16))) float so_[SPL][16][68];
    if (kg == 0) {
      sm_[w][n] = Mx;
      sl_[w][n] = Ls;
    }
#pragma unroll
    for (int nb = 0; nb < 4; nb++) *(v4f*)&so_[w][n][16 * nb + 4 * kg] = O[nb];
    __syncthreads();
    if (hd.done) return;
    for (int i = threadIdx.x; i < 16 * 16; i += 64 * SPL) {   // row i / 16, dims 4 (i % 16) ..
      const int r = i >> 4, d = 4 * (i & 15);
      if (t0 + r >= M) break;
      float mm = sm_[0][r];
#pragma unroll
      for (int k = 1; k < SPL; k++) mm = fmaxf(mm, sm_[k][r]);
      float l = 0.f;
      v4f o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < SPL; k++) {
        const float e = __builtin_amdgcn_exp2f(sm_[k][r] - mm);
        l += sl_[k][r] * e;
        o += *(const v4f*)&so_[k][r][d] * e;
      }
      gst((gu32x2*)(c.ao + (size_t)(t0 + r) * ILL_H + h * 64 + d),
          (gu32x2){f2h(o[0] / l) | (f2h(o[1] / l) << 16), f2h(o[2] / l) | (f2h(o[3] / l) << 16)});
    }
  }
}

// ---- commit ----------------------------------------------------------------------------
// Global argmax of rows lmh0 .. lmh0 + lmhn - 1 over the lm_head tiles, then the same
// commit as the pass kernel (greedy, chain or tree accept, KV compaction, State advance).
__global__ __launch_bounds__(ILL_WG_THREADS) void op_commit_kernel(IllPassArgs a, const uint64_t* amax, int ntiles, int kvswz) {
  __shared__ PassHdr H;
  __shared__ CommitLds C;
  __shared__ uint64_t best[16][ILL_WAVES];
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
  int stopreq = 0;   // the host's stop word (see ill_pass_kernel), waited for at the commit
  if (tid == 0 && a.stop_host) stopreq = __hip_atomic_load((const GAS int32_t*)a.stop_host, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  load_hdr(a, H);
  if (H.done) return;
  // the greatest key of a wave's lanes: the values first, then the lowest index among them
  auto wmax = [&](uint64_t k) {
    const uint32_t hi = (uint32_t)(k >> 32), m = group_reduce<64>(hi, OpMaxU{});
    return ((uint64_t)m << 32) | group_reduce<64>(hi == m ? (uint32_t)k : 0u, OpMaxU{});
  };
  auto of_row = [&](int t, int i0, int step) {   // tiles i0, i0 + step, .. of row t, four at a time
    const uint64_t* r = amax + (size_t)t * ntiles;
    uint64_t k = 0;
    for (int i = i0; i < ntiles; i += 4 * step) {
      uint64_t v[4];
#pragma unroll
      for (int u = 0; u < 4; u++) v[u] = gld(r + min(i + u * step, ntiles - 1));
#pragma unroll
      for (int u = 0; u < 4; u++) k = v[u] > k ? v[u] : k;
    }
    return wmax(k);
  };
  // one row: its tiles over all waves; more: a row per wave (16 rows: 25 us of commit with the
  // rows one after the other, each over all waves and through two barriers)
  const bool split = H.lmhn == 1;
  for (int t = H.lmh0 + (split ? 0 : w); t < H.lmh0 + H.lmhn; t += split ? 1 : ILL_WAVES) {
    const uint64_t k = split ? of_row(t, tid, ILL_WG_THREADS) : of_row(t, lane, 64);
    if (lane == 0) best[t][split ? w : 0] = k;
  }
  __syncthreads();
  if (tid < H.lmhn) {
    const int t = H.lmh0 + tid;
    uint64_t m = best[t][0];
    if (split)
      for (int i = 1; i < ILL_WAVES; i++) m = best[t][i] > m ? best[t][i] : m;
    C.g[t] = (int)(0xFFFFFFFFu - (uint32_t)(m & 0xFFFFFFFFu));
  }
  __syncthreads();
  commit_apply(a, H, C, false, stopreq, kvswz != 0);
}
