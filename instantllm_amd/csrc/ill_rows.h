// Row kernels: the layers of q8 and f16 passes of up to 16 rows (decode steps, verify passes,
// short prompts), five kernels per layer:
//   row_qkv_kernel   RMSNorm of x, QKV product, bias, RoPE, q and the K/V cache
//   row_attn_kernel  attention of a row's chunks of 512 positions, all heads of a KV group
//   row_o_kernel     the chunks' states combined, O product, x += ..
//   row_gu_kernel    RMSNorm of x, gate/up product, h = SiLU(gate) * up
//   row_down_kernel  down product, x += ..
// These passes move 0.8-17 MB per kernel and are bound by latency, not bandwidth: a kernel
// costs its launch (about 1.6 us in a graph), one or two memory round trips, and the
// instructions of one wave (1.7 ns each). So every kernel issues all of its loads at once (a
// wave holds its whole share of the weights in registers, K split over the waves of a
// workgroup and added in LDS in wave order), nothing is handed over as K-slice partials, and
// there is no kernel that only normalizes or adds: whoever updates x also leaves the sums of
// squares of its 16 columns (ssq), from which the next product's workgroups form the RMSNorm
// scale themselves.
//
// Measured against one kernel more per layer, with the gate/up and down products' K-slice
// partials in memory, the O projection inside attention and the residual sums and norms in
// kernels of their own (graph-replayed steps, us): q8 852 -> 591 after 512 positions, 970 ->
// 606 at 4000; f16 850 -> 656 and 969 -> 672; passes of 16 rows after 500 positions, q8, host
// clock, 1,294 -> 944. Kernel times of a q8 step at 512 positions: QKV 3.8, attention 6.8, O 3.8,
// gate/up 4.5, down 4.7 us.
//
// A row's arithmetic does not depend on the rows beside it or on MT (rows a workgroup holds):
// every output is the same MFMA sequence over K in the same order, and the attention's
// grouping depends on the row's own length only. So a row decoded alone and the same row in a
// 16-row pass give identical bits.
#pragma once
#include "ill_ops.h"

// Prompt chunks of up to this many rows run on the row kernels (16-row groups in grid.y, each
// reading the weights again), longer ones on the ring GEMMs, whose tiles share them. Whole
// prompts, ms, row kernels / ring: q4 48 tokens 0.78 / 1.12, 100 1.11 / 1.20, 128 1.22 / 1.22,
// 200 1.58 / 1.32; q8 100 1.10 / 1.23, 128 1.20 / 1.24, 200 1.52 / 1.33; f16 100 1.15 / 1.28,
// 128 1.26 / 1.30, 200 1.60 / 1.34.
#define ROW_MAXM 112
#define ROW_SSQ 64      // floats per row of the sum-of-squares partials (56 tiles, then zeros)
#define ROW_NSPLIT 8    // attention splits of a row: chunk c to split (c / 8) % 8, wave c % 8
#define ROW_ST 72       // floats per (row, head, split) state: o[64], m, l

// One k-step (64 columns) of a 16-row weight tile: lane (kg, n) holds row n, columns
// 16 kg .. + 15 (the tiled layout, op_wt_off: 1 KB (q8) or two runs of 1 KB (f16) per wave).
template <int FMT>
struct RowB {
  std::conditional_t<FMT == 2, uint2, uint4> q[FMT == 0 ? 2 : 1];
  std::conditional_t<FMT == 2, uint32_t, uint16_t> s;   // q8: the scale; q4: (scale, min)
};
template <int FMT>
__device__ __forceinline__ void row_fetch(const OpMat& W, int tile, int ks, int lane, RowB<FMT>& b) {
  const int blk = (tile >> 3) * (W.K >> 6) + ks, sub = tile & 7;
  if constexpr (FMT == 2) {
    b.q[0] = gld((const uint2*)(W.w + ((size_t)blk * 8 + sub) * 512) + lane);
    b.s = gld((const uint32_t*)W.s + (size_t)blk * 128 + sub * 16 + (lane & 15));
  } else if constexpr (FMT == 1) {
    b.q[0] = gld((const uint4*)(W.w + ((size_t)blk * 8 + sub) * 1024) + lane);
    const int per = 64 / W.qg;
    b.s = gld(W.s + ((size_t)blk * 128 + sub * 16 + (lane & 15)) * per + (per == 2 ? lane >> 5 : 0));
  } else {
    const uint4* p = (const uint4*)(W.w + ((size_t)blk * 8 + sub) * 2048);
    b.q[0] = gld(p + lane);
    b.q[1] = gld(p + 64 + lane);
  }
}
// columns 16 kg + 8 e .. + 7 as the MFMA operand
template <int FMT>
__device__ __forceinline__ v8h row_vals(const RowB<FMT>& b, int e) {
  if constexpr (FMT == 0) {
    return u4_to_v8h(b.q[e]);
  } else {
    v8h o;
    _Float16 h[8];
    if constexpr (FMT == 2) {
      op_q4x8(e == 0 ? b.q[0].x : b.q[0].y, (_Float16)h2f(b.s & 0xffff), (_Float16)h2f(b.s >> 16), h);
    } else {
      const _Float16 sc = (_Float16)h2f(b.s);
      op_q8x4(e == 0 ? b.q[0].x : b.q[0].z, sc, h);
      op_q8x4(e == 0 ? b.q[0].y : b.q[0].w, sc, h + 4);
    }
#pragma unroll
    for (int i = 0; i < 8; i++) o[i] = h[i];
    return o;
  }
}

// the rows a lane's operand and results hold: operand row n, result rows 4 kg + r
template <int MT>
__device__ __forceinline__ int row_a(int n) { return n & (MT - 1); }
// acc (lane (kg, n): rows 4 kg + r, column n) into red[row * 16 + n]
template <int MT>
__device__ __forceinline__ void row_put(float* red, const v4f& acc, int kg, int n) {
  if constexpr (MT == 16) {
#pragma unroll
    for (int r = 0; r < 4; r++) red[(4 * kg + r) * 16 + n] = acc[r];
  } else if (kg == 0) {
#pragma unroll
    for (int r = 0; r < MT; r++) red[r * 16 + n] = acc[r];
  }
}
__device__ __forceinline__ void row_wave_sync() {
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}
// RMSNorm scale of a row from this lane's sum-of-squares partial
__device__ __forceinline__ float row_scale(float part) {
  return __builtin_amdgcn_rsqf(gsum<64>(part) * (1.0f / (float)ILL_H) + ILL_EPS);
}

// Residual epilogue of row m, column 16 tile + i (thread (m, i) of 16-lane groups): x and the
// tile's sum of squares.
__device__ __forceinline__ void row_resid(const OpCtx& c, float* ssq, int m, int tile, int i, float x, float y) {
  const float v = x + y;
  gst(c.x + (size_t)m * ILL_H + 16 * tile + i, v);
  const float s = gsum<16>(v * v);
  if (i == 0) gst(ssq + (size_t)m * ROW_SSQ + tile, s);
}

// Embedding rows of the pass's tokens into x, with their sum-of-squares partials (a wave per row).
template <int FMT>
__global__ __launch_bounds__(256) void row_embed_kernel(OpCtx c, float* ssq, int M) {
  const int done = gld(&c.st->done);
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int t = blockIdx.x * 4 + w;
  if (t >= M) return;
  const int tok = gld(c.ptoks + t);
  float v[14];
#pragma unroll
  for (int i = 0; i < 14; i++) v[i] = op_dequant1<FMT>(c.emb, tok, 64 * i + lane);
  if (done) return;
#pragma unroll
  for (int i = 0; i < 14; i++) {
    gst(c.x + (size_t)t * ILL_H + 64 * i + lane, v[i]);
    const float s = gsum<16>(v[i] * v[i]);
    if ((lane & 15) == 0) gst(ssq + (size_t)t * ROW_SSQ + 4 * i + (lane >> 4), s);
  }
}

// QKV: a workgroup per rotary block (32 columns, two tiles), seven waves of two k-steps each.
// Wave w normalizes its own 128 columns of x.
template <int FMT, int MT>
__global__ __launch_bounds__(448) void row_qkv_kernel(OpCtx c, OpMat W, const float* gamma, const float* bias, const float* ssq,
                                                      int layer, int M, int pos_hint) {
  __shared__ __attribute__((aligned(16))) _Float16 As[7][MT][136];
  __shared__ float red[7][2][MT * 16];
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, kg = lane >> 4, n = lane & 15;
  const int b = blockIdx.x, m0 = 16 * blockIdx.y, Mg = min(M - m0, MT);
  float2 xv[MT];
  float sv[MT];
#pragma unroll
  for (int m = 0; m < MT; m++) {
    const int row = m0 + min(m, Mg - 1);
    sv[m] = gld(ssq + (size_t)row * ROW_SSQ + lane);
    xv[m] = gld((const float2*)(c.x + (size_t)row * ILL_H + 128 * w) + lane);
  }
  const float2 g = gld((const float2*)(gamma + 128 * w) + lane);
  const OpHdr hd = op_hdr(c);
  RowB<FMT> wb[2][2];
#pragma unroll
  for (int s = 0; s < 2; s++)
#pragma unroll
    for (int j = 0; j < 2; j++) row_fetch<FMT>(W, 2 * b + j, 2 * w + s, lane, wb[j][s]);
  // the epilogue's thread (em, ei): its bias values and the rotary row of the expected position
  const int em = min(tid >> 4, MT - 1), ei = tid & 15;
  float eb[2] = {gld(bias + 32 * b + ei), gld(bias + 32 * b + 16 + ei)};
  const int ep = min(pos_hint + m0 + em, c.maxctx - 1);
  const float2 cs = gld(c.rope + (size_t)ep * 32 + (b & 1) * 16 + ei);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int m = 0; m < MT; m++) {
    const float sc = row_scale(sv[m]);
    _Float16* d = &As[w][m][2 * lane];
    d[0] = (_Float16)__float2half(xv[m].x * sc * g.x);
    d[1] = (_Float16)__float2half(xv[m].y * sc * g.y);
  }
  row_wave_sync();
  v4f acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
  for (int s = 0; s < 2; s++)
#pragma unroll
    for (int e = 0; e < 2; e++) {
      const v8h a = *(const v8h*)&As[w][row_a<MT>(n)][64 * s + 16 * kg + 8 * e];
#pragma unroll
      for (int j = 0; j < 2; j++) acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, row_vals<FMT>(wb[j][s], e), acc[j], 0, 0, 0);
    }
#pragma unroll
  for (int j = 0; j < 2; j++) row_put<MT>(red[w][j], acc[j], kg, n);
  lds_barrier();
  if (hd.done || tid >= 16 * Mg) return;
  float x0 = red[0][0][tid], x1 = red[0][1][tid];
#pragma unroll
  for (int i = 1; i < 7; i++) {
    x0 += red[i][0][tid];
    x1 += red[i][1][tid];
  }
  epi_qkv(c, hd, layer, m0 + em, b, ei, x0, x1, ep, cs, eb);
}

// A row's output in two dims from its split states (o of the two dims; m, l), in split order.
__device__ __forceinline__ void row_combine(const float2* o, const float2* ml, int nne, float& y0, float& y1) {
  float mm = ml[0].x;
#pragma unroll
  for (int s = 1; s < ROW_NSPLIT; s++)
    if (s < nne) mm = fmaxf(mm, ml[s].x);
  float l = 0.f, a0 = 0.f, a1 = 0.f;
#pragma unroll
  for (int s = 0; s < ROW_NSPLIT; s++)
    if (s < nne) {
      const float e = att_exp(ml[s].x - mm);
      l = l + ml[s].y * e;
      a0 = a0 + o[s].x * e;
      a1 = a1 + o[s].y * e;
    }
  y0 = a0 / l;
  y1 = a1 / l;
}
// the splits of a row at pos + dep
__device__ __forceinline__ int row_splits(const OpCtx& c, int pos, int dep) {
  return __builtin_amdgcn_readfirstlane(min(ROW_NSPLIT, (row_chunks(pos, dep, c.maxctx) + 7) >> 3));
}

// Attention: a workgroup per (row, KV group, split j < nsplit) takes the splits j, j + nsplit, ..;
// wave w evaluates chunk 8 s + w (64 positions; then every 64th chunk) of split s for the
// group's seven heads at once: the heads are columns of the MFMA blocks (scores: K rows x heads,
// then V dims x heads), so K and V are read once per group, softmax statistics are per lane, and
// P needs no cross-lane move (the key of block b, row 4 kg + r is 32 (b / 2) + 8 kg + 4 (b % 2) + r,
// so a lane's scores are the eight consecutive keys of its operand slots). q and P enter
// the products as f16 pairs (high, low) that keep fp32's precision: q scaled by the power of two
// that brings the row and head's largest dim to f16's range, P by 2^15 and its low part by a
// further 2^11, into sums of its own. Unscaled pairs end in f16's subnormals (2^-25 absolute).
// Errors against 64 bits over the products' 2-norm, fp32 FMA chain / unscaled / these, in units of
// 2^-23: scores at |q| ~ 1, 0.1, 0.01: 1.2 / 1.4 / 0.8, 1.2 / 12 / 0.8, 1.2 / 121 / 0.8; P V with
// the scores spread over 5, 10 in log2: 1.2 / 4.6 / 0.7, 1.0 / 11 / 0.7. The scaling costs 0.5-1% of a
// pass (nine 1-row q8 steps 5.24 -> 5.29 ms after 500 positions, 5.50 -> 5.55 after 4000).
// The waves' states are combined in wave order into the split's state, the row's splits in split order: here with nsplit = 1 (c.ao gets the
// f16 output), else by the readers of att (row_o_kernel for one row, row_comb_kernel), with the
// same arithmetic, so the launch's split does not change the result.
// One chunk per wave up to 512 nsplit positions; 512 positions of 1 row take 2 workgroups. A graph
// keeps the nsplit of the context it was captured at; past it a wave takes several chunks, each
// next one streaming in from the current one's scores on (nine 1-row steps at 4000 positions captured
// at 8: q8 11.3 -> 10.1 ms, f16 11.9 -> 10.7; captured there 5.6 and 6.2).
// A tree pass's positions from pos on live in the slots of the row's ancestors (slot pos + row):
// K rows are loaded from those slots, V rows of such a chunk are patched in LDS.
template <bool SWZ>   // the K/V cache layout (ill_common.h): swizzled for q8 / f16, rows for q4
__global__ __launch_bounds__(64 * ILL_WAVES) void row_attn_kernel(OpCtx c, int layer, int M, int nsplit, float* att) {
  __shared__ float cm[ILL_WAVES][8], cl[ILL_WAVES][8];
  __shared__ __attribute__((aligned(16))) float co[ILL_WAVES][7][68];
  __shared__ int path[ILL_WAVES][16];
  __shared__ __attribute__((aligned(16))) uint16_t vst[2][64 * 72];   // (pass rows span two chunks at most)
  __shared__ float so[ROW_NSPLIT][7][64], sml[ROW_NSPLIT][7][2];      // nsplit 1: the splits' states
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, kg = lane >> 4, n = lane & 15;
  const int j = blockIdx.x % nsplit, g = (blockIdx.x / nsplit) % ILL_NKV, t = blockIdx.x / (nsplit * ILL_NKV);
  const float* qr = c.q + (size_t)t * ILL_H + (7 * g + min(n, 6)) * 64 + 8 * kg;
  float4 qf[2][2];
#pragma unroll
  for (int ks = 0; ks < 2; ks++) {
    qf[ks][0] = gld((const float4*)(qr + 32 * ks));
    qf[ks][1] = gld((const float4*)(qr + 32 * ks) + 1);
  }
  const OpHdr hd = op_hdr(c);
  const int tl = lane & 15;
  const int dp0 = gld(c.tree + ILL_TR_DEPTH + min(t, 15)), par = gld(c.tree + ILL_TR_PARENT + tl);
  const uint16_t* kb = c.kc + ((size_t)layer * ILL_NKV + g) * c.maxctx * 64;
  const uint16_t* vb = c.vt + ((size_t)layer * ILL_NKV + g) * c.maxctx * 64;
  uint4 kf[4][2], vf[4][2];
  auto kload = [&](int b, int slot) {
#pragma unroll
    for (int ks = 0; ks < 2; ks++) kf[b][ks] = gld((const uint4*)(kb + kv_k_off(slot, 32 * ks + 8 * kg, SWZ)));
  };
  auto kkey = [&](int b) { return 32 * (b >> 1) + 8 * (n >> 2) + 4 * (b & 1) + (n & 3); };
  auto vload = [&](int ch) {
#pragma unroll
    for (int nb = 0; nb < 4; nb++)
#pragma unroll
      for (int s = 0; s < 2; s++) vf[nb][s] = gld((const uint4*)(vb + kv_v_off(64 * ch + 32 * s + 8 * kg, 16 * nb + n, SWZ)));
  };
  // the first chunk at its plain slots, before the header is waited for
  {
    const int ch = min(8 * j + w, c.maxctx / 64 - 1);
#pragma unroll
    for (int b = 0; b < 4; b++) kload(b, 64 * ch + kkey(b));
    vload(ch);
  }
  __builtin_amdgcn_sched_barrier(0);
  // over the lane groups kg (the head's other keys or dims)
  auto over_kg = [](float v, auto op) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_int(v), __float_as_int(v), false, false);
    v = op(__int_as_float((int)a[0]), __int_as_float((int)a[1]));
    const auto q = __builtin_amdgcn_permlane32_swap(__float_as_int(v), __float_as_int(v), false, false);
    return op(__int_as_float((int)q[0]), __int_as_float((int)q[1]));
  };
  // q as f16 pairs of q 2^(15 - e), whose largest dim fills f16's range, and the power of two
  // that takes the scores back (with the 1 / 8)
  v8h qh[2], ql[2];
  float qback;
  {
    float v[2][8], mx = 0.f;
#pragma unroll
    for (int ks = 0; ks < 2; ks++) {
      const float x[8] = {qf[ks][0].x, qf[ks][0].y, qf[ks][0].z, qf[ks][0].w, qf[ks][1].x, qf[ks][1].y, qf[ks][1].z, qf[ks][1].w};
#pragma unroll
      for (int i = 0; i < 8; i++) {
        v[ks][i] = x[i];
        mx = fmaxf(mx, fabsf(x[i]));
      }
    }
    const int e = max(__builtin_amdgcn_frexp_expf(over_kg(mx, OpMaxF{})), -100);
    const float up = __builtin_ldexpf(1.f, 15 - e);
    qback = __builtin_ldexpf(0.125f, e - 15);
#pragma unroll
    for (int ks = 0; ks < 2; ks++)
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const float x = v[ks][i] * up;
        const _Float16 hi = (_Float16)x;
        qh[ks][i] = hi;
        ql[ks][i] = (_Float16)(x - (float)hi);
      }
  }
  const int pos = hd.pos;
  const bool tree = hd.mode == ILL_MODE_TREE;
  const int dep = tree ? dp0 : (hd.mode == ILL_MODE_DECODE ? 0 : t);
  const int L = pos + dep + 1, nch = row_chunks(pos, dep, c.maxctx);
  const int nne = min(ROW_NSPLIT, (nch + 7) >> 3);
  if (tree) {   // the row's ancestors by depth, from the parents held by lanes 0-15
    int pr = tl, r = __builtin_amdgcn_readfirstlane(t);
    for (int d = __builtin_amdgcn_readfirstlane(dep); d >= 0; --d) {
      if (tl == d) pr = r;
      r = r > 0 ? __builtin_amdgcn_readlane(par, r & 15) & 15 : 0;
    }
    if (lane < 16) path[w][lane] = pr;
    row_wave_sync();
  }
  auto slot_of = [&](int vp) { return min(vp < pos || !tree ? vp : pos + path[w][min(max(vp - pos, 0), 15)], c.maxctx - 1); };
#pragma unroll 1
  for (int s = j; s < nne; s += nsplit) {
    float Mx = -INFINITY, Ls = 0.f;
    v4f O[4];
#pragma unroll
    for (int nb = 0; nb < 4; nb++) O[nb] = (v4f){0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int ch = 8 * s + w; ch < nch; ch += 8 * ROW_NSPLIT) {
      const bool mixed = tree && 64 * ch + 63 >= pos;   // holds pass rows of a tree
      const int c1 = ch + 8 * ROW_NSPLIT, c2 = 8 * (s + nsplit) + w;   // the wave's next chunk: of this split, of its next one
      const int nx = c1 < nch ? c1 : s + nsplit < nne && c2 < nch ? c2 : -1;
      if (mixed && ch == 8 * j + w)   // (loaded from its plain slots)
#pragma unroll
        for (int b = 0; b < 4; b++) kload(b, slot_of(64 * ch + kkey(b)));
      if (mixed) {   // V: this wave's rows through LDS, positions pos .. L - 1 from the path's slots
        uint16_t* vr = vst[ch & 1];
#pragma unroll
        for (int nb = 0; nb < 4; nb++)
#pragma unroll
          for (int q = 0; q < 2; q++) *(uint4*)(vr + (16 * nb + n) * 72 + 32 * q + 8 * kg) = vf[nb][q];
        row_wave_sync();
        const int p0 = max(pos - 64 * ch, 0), p1 = min(L - 64 * ch, 64);
        uint16_t pv[16];
#pragma unroll
        for (int k = 0; k < 16; k++)
          if (p0 + k < p1) pv[k] = gld(vb + kv_v_off(slot_of(64 * ch + p0 + k), lane, SWZ));
#pragma unroll
        for (int k = 0; k < 16; k++)
          if (p0 + k < p1) vr[lane * 72 + p0 + k] = pv[k];
        row_wave_sync();
#pragma unroll
        for (int nb = 0; nb < 4; nb++)
#pragma unroll
          for (int q = 0; q < 2; q++) vf[nb][q] = *(const uint4*)(vr + (16 * nb + n) * 72 + 32 * q + 8 * kg);
      }
      if (64 * ch + 63 >= L) {   // positions past the row: values dropped (their probability is 0)
#pragma unroll
        for (int q = 0; q < 2; q++) {
          const int nv = L - (64 * ch + 32 * q + 8 * kg);
          uint32_t mk[4];
#pragma unroll
          for (int i = 0; i < 4; i++) mk[i] = nv >= 2 * i + 2 ? 0xffffffffu : (nv == 2 * i + 1 ? 0xffffu : 0u);
#pragma unroll
          for (int nb = 0; nb < 4; nb++) {
            vf[nb][q].x &= mk[0];
            vf[nb][q].y &= mk[1];
            vf[nb][q].z &= mk[2];
            vf[nb][q].w &= mk[3];
          }
        }
      }
      float sc[4][4];
      float mc = -INFINITY;
#pragma unroll
      for (int b = 0; b < 4; b++) {
        v4f d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < 2; ks++) {
          d = __builtin_amdgcn_mfma_f32_16x16x32_f16(u4_to_v8h(kf[b][ks]), qh[ks], d, 0, 0, 0);
          d = __builtin_amdgcn_mfma_f32_16x16x32_f16(u4_to_v8h(kf[b][ks]), ql[ks], d, 0, 0, 0);
        }
        const int vp = 64 * ch + 32 * (b >> 1) + 8 * kg + 4 * (b & 1);
#pragma unroll
        for (int r = 0; r < 4; r++) {
          sc[b][r] = vp + r < L ? d[r] * qback : -INFINITY;
          mc = fmaxf(mc, sc[b][r]);
        }
      }
      if (nx >= 0)   // the next chunk streams in from here, its values from the products with this one's on
#pragma unroll
        for (int b = 0; b < 4; b++) kload(b, slot_of(64 * nx + kkey(b)));
      mc = over_kg(mc, OpMaxF{});
      float lc = 0.f;
      v8h ph[2], pl[2];
#pragma unroll
      for (int b = 0; b < 4; b++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const float p = att_exp(sc[b][r] - mc), x = p * 32768.f;   // p <= 1
          lc += p;
          const _Float16 hi = (_Float16)x;
          ph[b >> 1][4 * (b & 1) + r] = hi;
          pl[b >> 1][4 * (b & 1) + r] = (_Float16)((x - (float)hi) * 2048.f);
        }
      lc = over_kg(lc, OpAddF{});
      const AttScale k = att_scale(Mx, mc);
      const float sb = k.sb * 0x1p-15f;
#pragma unroll
      for (int nb = 0; nb < 4; nb++) {
        v4f d = {0.f, 0.f, 0.f, 0.f}, dl = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < 2; q++) {
          d = __builtin_amdgcn_mfma_f32_16x16x32_f16(u4_to_v8h(vf[nb][q]), ph[q], d, 0, 0, 0);
          dl = __builtin_amdgcn_mfma_f32_16x16x32_f16(u4_to_v8h(vf[nb][q]), pl[q], dl, 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 4; r++) O[nb][r] = O[nb][r] * k.sa + fmaf(dl[r], 0x1p-11f, d[r]) * sb;
      }
      if (nx >= 0) vload(nx);
      Ls = att_fold(Ls, lc, k);
      Mx = k.mn;
    }
    if (n < 7) {
      if (kg == 0) {
        cm[w][n] = Mx;
        cl[w][n] = Ls;
      }
#pragma unroll
      for (int nb = 0; nb < 4; nb++) *(v4f*)&co[w][n][16 * nb + 4 * kg] = O[nb];
    }
    lds_barrier();
    if (w < 7 && !hd.done) {   // wave w: head w of the group, dim = lane
      float m[ILL_WAVES], l[ILL_WAVES], o[ILL_WAVES];
#pragma unroll
      for (int i = 0; i < ILL_WAVES; i++) {
        m[i] = cm[i][w];
        l[i] = cl[i][w];
        o[i] = co[i][w][lane];
      }
      float mo, lo, oo;
      att_combine<ILL_WAVES>(m, l, o, mo, lo, oo);
      if (nsplit > 1) {
        float* dst = att + (((size_t)t * ILL_NH + 7 * g + w) * ROW_NSPLIT + s) * ROW_ST;
        gst(dst + lane, oo);
        if (lane < 2) gst(dst + 64 + lane, lane == 0 ? mo : lo);
      } else {
        if (nne > 1) {
          so[s][w][lane] = oo;
          if (lane < 2) sml[s][w][lane] = lane == 0 ? mo : lo;
        }
        if (s + 1 == nne) {
          float l = lo, a0 = oo;
          if (nne > 1) {   // as row_combine, from LDS (this wave wrote the states)
            row_wave_sync();
            float mm = sml[0][w][0];
#pragma unroll 1
            for (int i = 1; i < nne; i++) mm = fmaxf(mm, sml[i][w][0]);
            l = a0 = 0.f;
#pragma unroll 1
            for (int i = 0; i < nne; i++) {
              const float e = att_exp(sml[i][w][0] - mm);
              l = l + sml[i][w][1] * e;
              a0 = a0 + so[i][w][lane] * e;
            }
          }
          const float y = a0 / l;
          gst((uint16_t*)(c.ao + (size_t)t * ILL_H + (7 * g + w) * 64 + lane), (uint16_t)__half_as_ushort(__float2half(y)));
        }
      }
    }
    if (s + nsplit < nne) lds_barrier();   // the states are read before the next split's are written
  }
}

// The split states of (row, head) pairs of passes of several rows, a wave per pair (lane: a
// dim), into c.ao.
__global__ __launch_bounds__(256) void row_comb_kernel(OpCtx c, const float* att, int M) {
  const int lane = threadIdx.x & 63, rh = 4 * blockIdx.x + (threadIdx.x >> 6);
  if (rh >= M * ILL_NH) return;
  const int t = rh / ILL_NH;
  const OpHdr hd = op_hdr(c);
  const int dp = gld(c.tree + ILL_TR_DEPTH + min(t, 15));
  const float* src = att + (size_t)rh * ROW_NSPLIT * ROW_ST;
  float2 o[ROW_NSPLIT], ml[ROW_NSPLIT];
#pragma unroll
  for (int s = 0; s < ROW_NSPLIT; s++) {   // (states past the row's splits are not used)
    o[s].x = gld(src + s * ROW_ST + lane);
    ml[s] = gld((const float2*)(src + s * ROW_ST + 64));
  }
  const int dep = hd.mode == ILL_MODE_TREE ? dp : (hd.mode == ILL_MODE_DECODE ? 0 : t);
  float y, unused;
  row_combine(o, ml, row_splits(c, hd.pos, dep), y, unused);
  if (!hd.done) gst((uint16_t*)(c.ao + (size_t)rh * 64 + lane), (uint16_t)__half_as_ushort(__float2half(y)));
}

// O projection: a workgroup per 16 output columns, seven waves of two k-steps (= heads) each.
// AO: rows m0 .., their f16 attention outputs in c.ao. Else one row from its split states: wave w
// combines those of its heads (lane: head 2 w + lane / 32, dims 2 (lane % 32), + 1). nsplit: the
// splits the host expects (loaded before the header is waited for; a longer row's others
// follow). Combining every row's states here as well took 16 us per layer at 16 rows (each of the
// 56 workgroups repeats it) against 4 + 3 with row_comb_kernel.
template <int FMT, int MT, bool AO>
__global__ __launch_bounds__(448) void row_o_kernel(OpCtx c, OpMat W, const float* att, float* ssq, int M, int nsplit) {
  __shared__ __attribute__((aligned(16))) _Float16 As[AO ? 1 : 7][1][136];
  __shared__ float red[7][MT * 16];
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, kg = lane >> 4, n = lane & 15;
  const int tile = blockIdx.x, m0 = AO ? 16 * blockIdx.y : 0, Mg = min(M - m0, MT);
  const OpHdr hd = op_hdr(c);
  RowB<FMT> wb[2];
  float ex;
  const int em = min(tid >> 4, MT - 1), ei = tid & 15;
  auto fetch = [&]() {
#pragma unroll
    for (int s = 0; s < 2; s++) row_fetch<FMT>(W, tile, 2 * w + s, lane, wb[s]);
    ex = gld(c.x + (size_t)(m0 + min(em, Mg - 1)) * ILL_H + 16 * tile + ei);
  };
  static_assert(AO || MT == 1, "several rows: from c.ao");
  uint4 av[AO ? 4 : 1];
  if constexpr (AO) {
    const uint4* ar = (const uint4*)(c.ao + (size_t)(m0 + min(n, Mg - 1)) * ILL_H + 128 * w);
#pragma unroll
    for (int i = 0; i < 4; i++) av[i] = gld(ar + 8 * (i >> 1) + 2 * kg + (i & 1));
    fetch();
    __builtin_amdgcn_sched_barrier(0);
  } else {
    const int h = 2 * w + (lane >> 5), d2 = 2 * (lane & 31);
    const float* st0 = att + (size_t)h * ROW_NSPLIT * ROW_ST;
    float2 o[ROW_NSPLIT], q[ROW_NSPLIT];   // (o of the two dims), (m, l)
    auto states = [&](int s0, int s1) {   // s0 <= s < s1
#pragma unroll
      for (int s = 0; s < ROW_NSPLIT; s++)
        if (s >= s0 && s < s1) {
          o[s] = gld((const float2*)(st0 + s * ROW_ST + d2));
          q[s] = gld((const float2*)(st0 + s * ROW_ST + 64));
        }
    };
    states(0, nsplit);
    fetch();
    const int dp = gld(c.tree + ILL_TR_DEPTH);
    __builtin_amdgcn_sched_barrier(0);
    const int nne = row_splits(c, hd.pos, hd.mode == ILL_MODE_TREE ? dp : 0);
    if (nne > nsplit) states(nsplit, nne);
    float y0, y1;
    row_combine(o, q, nne, y0, y1);
    _Float16* d = &As[w][0][2 * lane];   // k-step lane / 32, column 2 (lane % 32)
    d[0] = (_Float16)__float2half(y0);
    d[1] = (_Float16)__float2half(y1);
    row_wave_sync();
  }
  v4f acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < 2; s++)
#pragma unroll
    for (int e = 0; e < 2; e++) {
      v8h a;
      if constexpr (AO) a = u4_to_v8h(av[2 * s + e]);
      else a = *(const v8h*)&As[w][row_a<MT>(n)][64 * s + 16 * kg + 8 * e];
      acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, row_vals<FMT>(wb[s], e), acc, 0, 0, 0);
    }
  row_put<MT>(red[w], acc, kg, n);
  lds_barrier();
  if (hd.done || tid >= 16 * Mg) return;
  float y = red[0][tid];
#pragma unroll
  for (int i = 1; i < 7; i++) y += red[i][tid];
  row_resid(c, ssq, m0 + em, tile, ei, ex, y);
}

// Gate/up: a workgroup per four tiles (32 hidden units), a pair of waves per tile splitting K.
// The workgroup normalizes the rows once into LDS.
template <int FMT, int MT>
__global__ __launch_bounds__(512) void row_gu_kernel(OpCtx c, OpMat W, const float* gamma, const float* ssq, int M) {
  __shared__ __attribute__((aligned(16))) _Float16 As[MT][ILL_H + 8];
  __shared__ float red[2][4][MT * 16];
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, kg = lane >> 4, n = lane & 15;
  const int wt = w >> 1, wk = w & 1, tile = 4 * blockIdx.x + wt;
  const int m0 = 16 * blockIdx.y, Mg = min(M - m0, MT);
  const int done = gld(&c.st->done);
  const int k2 = min(tid, 447);   // columns 2 k2, + 1
  constexpr int MB = MT < 4 ? MT : 4;   // rows normalized per round
  float2 xv[MB];
  float sv[MB];
  auto rows = [&](int r0) {
#pragma unroll
    for (int m = 0; m < MB; m++) {
      const int row = m0 + min(r0 + m, Mg - 1);
      sv[m] = gld(ssq + (size_t)row * ROW_SSQ + lane);
      xv[m] = gld((const float2*)(c.x + (size_t)row * ILL_H) + k2);
    }
  };
  rows(0);
  const float2 g = gld((const float2*)gamma + k2);
  RowB<FMT> wb[7];
#pragma unroll
  for (int s = 0; s < 7; s++) row_fetch<FMT>(W, tile, 7 * wk + s, lane, wb[s]);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int r0 = 0; r0 < MT; r0 += MB) {
    if (r0 > 0) {
      if (r0 >= Mg) break;
      rows(r0);
    }
#pragma unroll
    for (int m = 0; m < MB; m++) {
      const float sc = row_scale(sv[m]);
      if (tid < 448) {
        _Float16* d = &As[r0 + m][2 * tid];
        d[0] = (_Float16)__float2half(xv[m].x * sc * g.x);
        d[1] = (_Float16)__float2half(xv[m].y * sc * g.y);
      }
    }
  }
  lds_barrier();
  v4f acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < 7; s++)
#pragma unroll
    for (int e = 0; e < 2; e++) {
      const v8h a = *(const v8h*)&As[row_a<MT>(n)][64 * (7 * wk + s) + 16 * kg + 8 * e];
      acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, row_vals<FMT>(wb[s], e), acc, 0, 0, 0);
    }
  row_put<MT>(red[wk][wt], acc, kg, n);
  lds_barrier();
  // thread (tile, row, unit): gate and up columns g, g, u, u of each four
  const int et = MT == 16 ? tid >> 7 : tid / (8 * MT), em = (tid >> 3) & (MT - 1), u = tid & 7;
  if (done || et >= 4 || em >= Mg) return;
  const int col = em * 16 + 4 * (u >> 1) + (u & 1);
  const float gv = red[0][et][col] + red[1][et][col], uv = red[0][et][col + 2] + red[1][et][col + 2];
  epi_silu(c, m0 + em, 8 * (4 * blockIdx.x + et) + u, gv, uv);
}

// Down projection: a workgroup per 16 output columns, sixteen waves of four or five k-steps.
template <int FMT, int MT>
__global__ __launch_bounds__(1024) void row_down_kernel(OpCtx c, OpMat W, float* ssq, int M) {
  constexpr int NW = 16, NK = 5, KS = ILL_FF / 64;
  __shared__ __attribute__((aligned(16))) _Float16 As[MT <= 4 ? NW : 1][MT <= 4 ? MT : 1][64 * NK + 8];
  __shared__ float red[NW][MT * 16];
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, kg = lane >> 4, n = lane & 15;
  const int tile = blockIdx.x, m0 = 16 * blockIdx.y, Mg = min(M - m0, MT);
  const int done = gld(&c.st->done);
  const int k0 = w * KS / NW, ns = (w + 1) * KS / NW - k0;   // 4 or 5
  // A: up to 4 rows, the wave's columns of each row through LDS; more rows, straight into the operand
  uint4 av[MT <= 4 ? MT : 2 * NK];
  if constexpr (MT <= 4) {
#pragma unroll
    for (int m = 0; m < MT; m++)
      av[m] = gld((const uint4*)(c.h + (size_t)(m0 + min(m, Mg - 1)) * ILL_FF + 64 * k0) + min(lane, 8 * ns - 1));
  } else {
    const uint4* hr = (const uint4*)(c.h + (size_t)(m0 + min(n, Mg - 1)) * ILL_FF);
#pragma unroll
    for (int s = 0; s < NK; s++)
#pragma unroll
      for (int e = 0; e < 2; e++) av[2 * s + e] = gld(hr + 8 * (k0 + min(s, ns - 1)) + 2 * kg + e);
  }
  RowB<FMT> wb[NK];
#pragma unroll
  for (int s = 0; s < NK; s++) row_fetch<FMT>(W, tile, k0 + min(s, ns - 1), lane, wb[s]);
  const int em = min(tid >> 4, MT - 1), ei = tid & 15;
  const float ex = gld(c.x + (size_t)(m0 + min(em, Mg - 1)) * ILL_H + 16 * tile + ei);
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (MT <= 4) {
#pragma unroll
    for (int m = 0; m < MT; m++)
      if (lane < 8 * NK) *(uint4*)&As[w][m][8 * lane] = av[m];
    row_wave_sync();
  }
  v4f acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < NK; s++)
    if (s < ns) {
#pragma unroll
      for (int e = 0; e < 2; e++) {
        v8h a;
        if constexpr (MT <= 4) a = *(const v8h*)&As[w][row_a<MT>(n)][64 * s + 16 * kg + 8 * e];
        else a = u4_to_v8h(av[2 * s + e]);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, row_vals<FMT>(wb[s], e), acc, 0, 0, 0);
      }
    }
  row_put<MT>(red[w], acc, kg, n);
  lds_barrier();
  if (done || tid >= 16 * Mg) return;
  float y = red[0][tid];
#pragma unroll
  for (int i = 1; i < NW; i++) y += red[i][tid];
  row_resid(c, ssq, m0 + em, tile, ei, ex, y);
}
