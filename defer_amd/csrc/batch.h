// batch.h -- the batched forward: B rows, each a (cache, position, token),
// step through the model together and every matrix product is an MFMA GEMM.
//
// Batch invariance. Every output element of every matrix product is computed
// in the one order the one-token path uses (device.h, "Row dot products"):
// 16 segments s, segment s holding the elements 64*i + 4*s + c (i
// ascending, c = 0..3), each segment a chain of fused multiply-adds from +0,
// then the complete binary tree over the 16 segment sums.
// v_mfma_f32_16x16x4_f32 computes, for each output, exactly
// fma(a3,b3,fma(a2,b2,fma(a1,b1,fma(a0,b0,c)))) -- four links of such a
// chain -- so chaining one MFMA per chunk reproduces a segment's sum bit for
// bit, and the tree is then formed from the 16 segment accumulators. The
// result of a row depends on that row's inputs only: not on B, not on the
// other rows, not on the tiling. Everything else a row goes through
// (RMSNorm, RoPE, attention, combine, residuals, activation, sampling) runs
// the same expressions as the one-token path, or the very same functions.
#pragma once

#include "phases.h"

namespace dg {

typedef float f4v __attribute__((ext_vector_type(4)));

// ------------------------------------------------------------ panel layout
//
// GEMM operands are stored as panels: a matrix of R rows and K columns
// becomes [ceil(R/16)][nch = ceil(K/64)][4 quarters][64 lanes][4 floats],
// float u of quarter q of lane l = r + 16c in chunk i of tile T holding
// element (16*T + r, 64*i + 4*(4q + u) + c), zero outside the matrix. Lane l's
// float u of quarter q is its MFMA operand (A for weights, B for activations)
// of segment 4q + u; a (tile, chunk) is 4 KB, each quarter 1 KB contiguous,
// so one 16-byte-per-lane load moves a quarter, and lanes read LDS copies of
// it at consecutive addresses.

constexpr uint32_t PANEL_TILE = 1024;  // floats per (16-row tile, chunk)

__host__ __device__ inline uint32_t panel_chunks(uint32_t K) { return (K + 63) / 64; }
__host__ __device__ inline size_t panel_floats(uint32_t R, uint32_t K) {
  return (size_t)((R + 15) / 16) * panel_chunks(K) * PANEL_TILE;
}

// Position of element (row r, column k) in a panel of nch chunks.
__host__ __device__ inline size_t panel_at(uint32_t r, uint32_t k, uint32_t nch) {
  const uint32_t i = k / 64, s = (k % 64) / 4, c = k % 4;
  return (((size_t)(r / 16) * nch + i) * 4 + s / 4) * 256 + ((r % 16) + 16 * c) * 4 + s % 4;
}

// Rows [0, R0) from src0, rows [R0, R) from src1 (row r - R0): a stacked
// matrix without a stacked copy. ld: row stride of both sources.
__global__ void k_to_panel(const float* __restrict__ src0, const float* __restrict__ src1,
                           uint32_t R0, uint32_t R, uint32_t K, uint32_t ld,
                           float* __restrict__ dst) {
  const size_t n = panel_floats(R, K);
  const uint32_t nch = panel_chunks(K);
  for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < n;
       e += (size_t)gridDim.x * blockDim.x) {
    const uint32_t u = (uint32_t)(e % 4), l = (uint32_t)((e / 4) % 64),
                   q = (uint32_t)((e / 256) % 4);
    const size_t rest = e / PANEL_TILE;
    const uint32_t i = (uint32_t)(rest % nch);
    const size_t r = (rest / nch) * 16 + l % 16;
    const uint32_t k = 64 * i + 4 * (4 * q + u) + l / 16;
    float v = 0.0f;
    if (r < R && k < K) v = r < R0 ? src0[r * ld + k] : src1[(r - R0) * ld + k];
    dst[e] = v;
  }
}

// ------------------------------------------------------------------ GEMM

enum GemmOut : uint32_t {
  GO_PLAIN = 0,  // Y[b][o] = y
  GO_RESID = 1,  // Y[b][o] = Y[b][o] + y   (the residual stream, in place; also into panel P)
  GO_TAG = 2,    // T[b][o] = tag(gen[b], inv[b] * y)  (tagged logits)
  // Outputs of a pair of rows, W the pairs' first rows and their partners
  // stacked in blocks of `blk` row tiles (see GemmOutArgs):
  GO_ACT = 3,    // P[b][o] = act(gate * inv[b]) * (up * inv[b])  (phase_gu)
  GO_QKV = 4,    // rotated q to qf[b][q], k and v to the row's cache (phase_qkv)
};
constexpr bool gemm_pairs(uint32_t out) { return out == GO_ACT || out == GO_QKV; }

// One row of a batch: the cache it extends, at which position and
// generation base, with which token.
struct BRow {
  float* kc;
  float* vc;
  uint32_t cap, pos, tick, token;
};

// Where a product goes. A pair product's row tiles come in pairs: pair p is
// tile p / blk * 2 * blk + p % blk and the one blk later (gate and up rows:
// blk = all the gate tiles; the two halves of each rotated head: blk = half a
// head).
struct GemmOutArgs {
  float* Y;             // GO_PLAIN, GO_RESID, GO_TAG (u64 words): [B][ldy]
  uint32_t ldy;
  float* P;             // GO_RESID (K = M), GO_ACT (K = M / 2): panel of the output
  const float* inv;     // GO_TAG, GO_ACT, GO_QKV: the rows' 1/rms
  const uint32_t* gen;  // GO_TAG
  uint32_t blk;         // pair products
  uint32_t act;         // GO_ACT
  const float* X;       // GO_ACT, at most 16 rows: form 1/rms from the rows [B][K] instead of inv
  float eps;
  // GO_QKV
  const BRow* rows;
  const float2* rope;
  const float* bias;    // or null
  float* qf;
  uint32_t l, hd, half, nh, nkv, kvs;
};

// 1/rms of N rows of n floats, by one wave: lane partials over the float4s
// at 4*lane + 256*i (i ascending), then the wave tree. The rows' loads and
// chains run side by side.
template <int N>
__device__ __forceinline__ void rms_rows_inv(const float* const (&x)[N], uint32_t n, float eps,
                                             uint32_t lane, float (&inv)[N]) {
  float ss[N];
#pragma unroll
  for (int r = 0; r < N; ++r) ss[r] = 0.0f;
  for (uint32_t j = lane * 4; j < n; j += 256) {
    float4 v[N];
#pragma unroll
    for (int r = 0; r < N; ++r) v[r] = *reinterpret_cast<const float4*>(x[r] + j);
#pragma unroll
    for (int r = 0; r < N; ++r) {
      ss[r] = fmaf(v[r].x, v[r].x, ss[r]);
      ss[r] = fmaf(v[r].y, v[r].y, ss[r]);
      ss[r] = fmaf(v[r].z, v[r].z, ss[r]);
      ss[r] = fmaf(v[r].w, v[r].w, ss[r]);
    }
  }
  wave_sum_n<N>(ss);
#pragma unroll
  for (int r = 0; r < N; ++r) inv[r] = 1.0f / sqrtf(ss[r] / (float)n + eps);
}
__device__ __forceinline__ float rms_row_inv(const float* __restrict__ x, uint32_t n, float eps,
                                             uint32_t lane) {
  const float* const p[1] = {x};
  float inv[1];
  rms_rows_inv(p, n, eps, lane, inv);
  return inv[0];
}

// 16 bytes at a byte offset from a wave-uniform base.
__device__ __forceinline__ float4 ldg4_at(const float* base, uint32_t byte_off) {
  const v4f x = *(const AS_GLOBAL v4f*)((const AS_GLOBAL char*)(uintptr_t)base + byte_off);
  return make_float4(x.x, x.y, x.z, x.w);
}

// The order of a launch's tasks, rows (row groups) x cols (column groups):
// the dispatcher deals workgroups to the XCDs in turn, so workgroup b runs
// task b / NXCD of a contiguous run of XCD b % NXCD, and the runs go through
// bands of `band` column groups, row group by row group. What an XCD has in
// flight is then a block of a few row groups by a band: a weight tile is
// fetched into its L2 once per band, not once per column group (8B shape,
// 28672 x 4096 by 500 rows: 1,368 us with the rows fastest, 1,013 so).
struct TaskXY {
  uint32_t x, y;
};
__device__ __forceinline__ TaskXY gemm_task(uint32_t b, uint32_t n, uint32_t rows, uint32_t cols,
                                            uint32_t band) {
  const uint32_t k = b % NXCD, t = k * (n / NXCD) + min(k, n % NXCD) + b / NXCD;
  const uint32_t c0 = t / (rows * band) * band, w = min(band, cols - c0), r = t - rows * c0;
  return {r / w, c0 + r % w};
}

// Y[b][o] = W[o] . X[b] for o < M, b < B, K columns. A task is TR row tiles
// by TC column tiles; its four waves take a quarter of the segments each
// (wave q: segments 4q .. 4q+3, quarter q of every panel tile, 1 KB
// contiguous), so every operand byte is used by one wave only: it goes from
// memory straight into that wave's registers, D chunks ahead of its use, and
// the main loop has neither LDS nor barriers. Each wave forms its quarter's
// subtree of tree16, ((s_4q + s_4q+1) + (s_4q+2 + s_4q+3)); the four meet in
// LDS as (t_0 + t_1) + (t_2 + t_3) -- the complete tree over the 16 segments
// -- and the output is written from there.
//
// Bound: the matrix cores for wide batches (two 4x2 workgroups per CU, one
// wave of each per SIMD), memory for narrow ones. Measured against the
// operands shared through LDS (one workgroup of eight waves, a barrier per
// chunk), us before -> now: 3072 x 576 by 2048 rows 86 -> 75 (97 TFLOP/s),
// 576 x 1536 by 2048 59 -> 38, 576 x 1536 by 301 35 -> 9.2, 28672 x 4096 by
// 500 1,338 -> 1,013 (116 TFLOP/s), 128256 x 4096 by 1 row 1,042 -> 342
// (6.1 TB/s of weights). Workgroups that take several tasks and load ahead
// across them measured the same or slower.
constexpr uint32_t GEMM_BAND = 32;  // column tiles of a band
__host__ __device__ constexpr int gemm_depth(int tr, int tc) { return tr * tc >= 8 ? 2 : tr * tc >= 4 ? 3 : 4; }
template <int TR, int TC, uint32_t OUT, bool PARTIAL>
__global__ __launch_bounds__(256, 2) void k_gemm(const float* __restrict__ Wp, uint32_t M, uint32_t K,
                                                 const float* __restrict__ Xp, uint32_t B,
                                                 const GemmOutArgs out) {
  constexpr int D = gemm_depth(TR, TC), NT = TR * TC;
  __shared__ float4 sub[4 * NT * WAVE];  // [quarter][tile][lane]
  // The wave index is uniform: scalar registers for it and the tile bases.
  const uint32_t q = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE;
  const uint32_t nch = panel_chunks(K), nrt = (M + 15) / 16, nct = (B + 15) / 16;
  const TaskXY task = gemm_task(blockIdx.x, gridDim.x, (nrt + TR - 1) / TR, (nct + TC - 1) / TC, GEMM_BAND / TC);
  // Row tile r of the task. Tiles past the last one load a real tile, never
  // used.
  auto row_tile = [&](uint32_t r) {
    if (!gemm_pairs(OUT)) return TR * task.x + r;
    constexpr uint32_t HT = TR >= 2 ? TR / 2 : 1;
    const uint32_t p = HT * task.x + r % HT;
    return p / out.blk * 2 * out.blk + p % out.blk + (r < HT ? 0 : out.blk);
  };
  const float *wa[TR], *xb[TC];
#pragma unroll
  for (int r = 0; r < TR; ++r)
    wa[r] = Wp + (size_t)min(row_tile(r), nrt - 1) * nch * PANEL_TILE + q * 256;
#pragma unroll
  for (int c = 0; c < TC; ++c)
    xb[c] = Xp + (size_t)min(TC * task.y + c, nct - 1) * nch * PANEL_TILE + q * 256;
  f4v acc[TR][TC][4];
#pragma unroll
  for (int r = 0; r < TR; ++r)
#pragma unroll
    for (int c = 0; c < TC; ++c)
#pragma unroll
      for (int u = 0; u < 4; ++u) acc[r][c][u] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
  float4 a[D][TR], b[D][TC];
  const uint32_t last = (nch - 1) * (PANEL_TILE * 4) + lane * 16;
  uint32_t off = lane * 16;
  auto load = [&](int d) {  // the next chunk (past the last one: that one again, never used)
#pragma unroll
    for (int r = 0; r < TR; ++r) a[d][r] = ldg4_at(wa[r], off);
#pragma unroll
    for (int c = 0; c < TC; ++c) b[d][c] = ldg4_at(xb[c], off);
    off = min(off + PANEL_TILE * 4, last);
  };
  auto mfma = [&](int d, int u) {
#pragma unroll
    for (int r = 0; r < TR; ++r)
#pragma unroll
      for (int c = 0; c < TC; ++c)
        acc[r][c][u] = __builtin_amdgcn_mfma_f32_16x16x4f32((&a[d][r].x)[u], (&b[d][c].x)[u],
                                                            acc[r][c][u], 0, 0, 0);
  };
#pragma unroll
  for (int d = 0; d < D; ++d) load(d);
  // What the outputs need from memory: the small tasks request it here, so
  // that its latency does not follow the main loop's (18 steps of 7 sessions,
  // 135M shape: 29.3 -> 28.8 ms); the large ones after the loop (1 % faster
  // there: registers, and another workgroup's MFMAs to wait behind).
  constexpr bool EARLY = NT <= 2;
  // Pair products: one pair per wave, pair p, column bc of each lane.
  const uint32_t p = TR / 2 * task.x + q / TC, pbc = (TC * task.y + q % TC) * 16 + lane % 16;
  const bool pair_out = gemm_pairs(OUT) && q < NT / 2 && 2 * p < nrt && pbc < B;
  float iv = 0.0f;
  BRow row;
  uint32_t hb = 0, hi = 0;  // head block, first of the lane's four elements in its first half
  float4 cs[2];
  auto pair_inputs = [&]() {
    if (!pair_out) return;
    if (!(OUT == GO_ACT && out.X)) iv = out.inv[pbc];
    if (OUT == GO_QKV) {
      row = out.rows[pbc];
      hb = p / out.blk;
      hi = p % out.blk * 16 + 4 * (lane / 16);
      const float4* rp = reinterpret_cast<const float4*>(out.rope + (size_t)row.pos * out.half + hi);
      cs[0] = rp[0];
      cs[1] = rp[1];
    }
  };
  // Other products: tiles q, q + 4, ...; the residual's old values.
  constexpr int NO = gemm_pairs(OUT) ? 1 : (NT + 3) / 4;
  struct OutAt {
    uint32_t bc, o;
    bool on, vec;  // in range; four outputs inside M and 16-byte aligned
  };
  auto out_at = [&](int k) {
    const uint32_t t = 4 * k + q, T = TR * task.x + t / TC;
    OutAt r;
    r.bc = (TC * task.y + t % TC) * 16 + lane % 16;
    r.o = T * 16 + 4 * (lane / 16);
    r.on = t < NT && T < nrt && r.bc < B;
    r.vec = OUT != GO_TAG && r.o + 4 <= M && (((size_t)r.bc * out.ldy + r.o) & 3) == 0;
    return r;
  };
  float4 old[NO];
  auto old_values = [&]() {
#pragma unroll
    for (int k = 0; k < NO; ++k) {
      const OutAt r = out_at(k);
      if (r.on && r.vec) old[k] = *reinterpret_cast<const float4*>(out.Y + (size_t)r.bc * out.ldy + r.o);
    }
  };
  // Few rows: every workgroup forms their 1/rms itself (wave q: rows 4q ..),
  // a third more bytes from L2 than its operands but no launch of its own
  // before this product: 2.6 us per layer of 7 rows (135M shape).
  __shared__ float row_inv[16];
  if (OUT == GO_ACT && TC == 1 && out.X) {
    const float* xr[4];
    float ri[4];
#pragma unroll
    for (uint32_t u = 0; u < 4; ++u) xr[u] = out.X + (size_t)min(4 * q + u, B - 1) * K;
    rms_rows_inv(xr, K, out.eps, lane, ri);
    if (lane < 4) row_inv[4 * q + lane] = lane == 0 ? ri[0] : lane == 1 ? ri[1] : lane == 2 ? ri[2] : ri[3];
  }
  if (EARLY) {
    if (gemm_pairs(OUT)) pair_inputs();
    if (OUT == GO_RESID) old_values();
  }
  const uint32_t nfull = K / 64;
  uint32_t i = 0;
  for (; i + D <= nfull; i += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
#pragma unroll
      for (int u = 0; u < 4; ++u) mfma(d, u);
      load(d);
    }
  }
#pragma unroll
  for (int d = 0; d < D; ++d) {
    if (i + d < nfull) {
#pragma unroll
      for (int u = 0; u < 4; ++u) mfma(d, u);
    } else if (PARTIAL && i + d < nch) {
      // A last, partial chunk: the segments past K are left alone (their
      // zero padding would still turn a -0 sum into +0).
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (64 * nfull + 4 * (4 * q + u) < K) mfma(d, u);
    }
  }
#pragma unroll
  for (int r = 0; r < TR; ++r)
#pragma unroll
    for (int c = 0; c < TC; ++c) {
      const f4v t = (acc[r][c][0] + acc[r][c][1]) + (acc[r][c][2] + acc[r][c][3]);
      sub[(q * NT + r * TC + c) * WAVE + lane] = make_float4(t[0], t[1], t[2], t[3]);
    }
  __syncthreads();
  // Tile t's outputs: rows 4*(lane/16) .. +3, column lane % 16.
  auto total = [&](uint32_t t, float (&v)[4]) {
    float4 s[4];
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) s[k] = sub[(k * NT + t) * WAVE + lane];
    v[0] = (s[0].x + s[1].x) + (s[2].x + s[3].x);
    v[1] = (s[0].y + s[1].y) + (s[2].y + s[3].y);
    v[2] = (s[0].z + s[1].z) + (s[2].z + s[3].z);
    v[3] = (s[0].w + s[1].w) + (s[2].w + s[3].w);
  };
  if constexpr (gemm_pairs(OUT)) {
    static_assert(NT / 2 <= 4 && TR % 2 == 0, "a pair of tiles per wave");
    if (!pair_out) return;
    if (!EARLY) pair_inputs();
    float y0[4], y1[4];
    total(q, y0);
    total(NT / 2 + q, y1);
    if (OUT == GO_ACT) {
      if (TC == 1 && out.X) iv = row_inv[lane % 16];
      const uint32_t nchp = panel_chunks(M / 2), o = p * 16 + 4 * (lane / 16);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        out.P[panel_at(pbc, o + j, nchp)] = act_fn(y0[j] * iv, out.act) * (y1[j] * iv);
    } else {
      // phase_qkv's epilogue (QkvEpiPair's expressions) of four pairs.
      const bool rotated = hb < out.nh + out.nkv;
      const float* bias = out.bias ? out.bias + hb * out.hd + hi : nullptr;
      float a0[4], a1[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float e0 = bias ? bias[j] : 0.0f, e1 = bias ? bias[out.half + j] : 0.0f;
        y0[j] = y0[j] * iv + e0;
        y1[j] = y1[j] * iv + e1;
        a0[j] = y0[j];
        a1[j] = y1[j];
        if (rotated) {
          const float cx = (&cs[j / 2].x)[j % 2 * 2], cy = (&cs[j / 2].x)[j % 2 * 2 + 1];
          a0[j] = y0[j] * cx - y1[j] * cy;
          a1[j] = y1[j] * cx + y0[j] * cy;
        }
      }
      float* dst;
      if (hb < out.nh) {
        dst = out.qf + ((size_t)pbc * out.nh + hb) * out.hd;
      } else {
        const uint32_t gi = rotated ? hb - out.nh : hb - out.nh - out.nkv;
        dst = (rotated ? row.kc : row.vc) + (((size_t)out.l * out.nkv + gi) * row.cap + row.pos) * out.kvs;
      }
      *reinterpret_cast<float4*>(dst + hi) = make_float4(a0[0], a0[1], a0[2], a0[3]);
      *reinterpret_cast<float4*>(dst + hi + out.half) = make_float4(a1[0], a1[1], a1[2], a1[3]);
    }
    return;
  }
  if (!EARLY && OUT == GO_RESID) old_values();
#pragma unroll
  for (int k = 0; k < NO; ++k) {
    const OutAt r = out_at(k);
    if (!r.on) continue;
    const uint32_t bc = r.bc, o = r.o;
    float v[4];
    total(4 * k + q, v);
    float* Y = out.Y;
    const size_t at = (size_t)bc * out.ldy + o;
    const uint32_t nchp = panel_chunks(M);  // the residual's panel: K = M
    if (r.vec) {
      float4 w = make_float4(v[0], v[1], v[2], v[3]);
      if (OUT == GO_RESID) {
        w = make_float4(old[k].x + v[0], old[k].y + v[1], old[k].z + v[2], old[k].w + v[3]);
        out.P[panel_at(bc, o, nchp)] = w.x;
        out.P[panel_at(bc, o + 1, nchp)] = w.y;
        out.P[panel_at(bc, o + 2, nchp)] = w.z;
        out.P[panel_at(bc, o + 3, nchp)] = w.w;
      }
      *reinterpret_cast<float4*>(Y + at) = w;
      continue;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (o + j >= M) continue;
      if (OUT == GO_PLAIN) {
        Y[at + j] = v[j];
      } else if (OUT == GO_RESID) {
        const float w = Y[at + j] + v[j];
        Y[at + j] = w;
        out.P[panel_at(bc, o + j, nchp)] = w;
      } else {
        reinterpret_cast<u64*>(Y)[at + j] =
            ((u64)out.gen[bc] << 32) | (u64)__float_as_uint(out.inv[bc] * v[j]);
      }
    }
  }
}

// ------------------------------------------------------------- rows

// X[b] = E[token_b] (model.rs:428), and its panel XP; token_b from dtok
// (device, e.g. just sampled) when given, else from the row.
__global__ void k_b_embed(const BRow* __restrict__ rows, const uint32_t* __restrict__ dtok,
                          const float* __restrict__ embed, uint32_t h,
                          float* __restrict__ X, float* __restrict__ XP) {
  const uint32_t b = blockIdx.x, nch = panel_chunks(h);
  const float* e = embed + (size_t)(dtok ? dtok[b] : rows[b].token) * h;
  for (uint32_t i = threadIdx.x; i < h; i += blockDim.x) {
    const float v = e[i];
    X[(size_t)b * h + i] = v;
    XP[panel_at(b, i, nch)] = v;
  }
}

// inv[b] = 1/rms(X[b]) in the order of rms_inv: each lane's elements
// 4*lane + 256*k ascending, then wave_sum. One wave per row.
__global__ __launch_bounds__(256) void k_b_rms(const float* __restrict__ X, uint32_t B, uint32_t n,
                                               float eps, float* __restrict__ inv) {
  const uint32_t b = blockIdx.x * 4 + threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
  if (b >= B) return;
  const float r = rms_row_inv(X + (size_t)b * n, n, eps, lane);
  if (lane == 0) inv[b] = r;
}

// QKV epilogue of the one-token path (phase_qkv) for pair i of head block
// hb of a batch row at position pos: the product's rows r0 = hb * hd + i and
// r1 = r0 + half (y: the row's product), scaled by the row's 1/rms, biased,
// and rotated (q and k heads) -- phase_qkv's expressions. load() reads what
// it needs from memory, value() computes.
struct QkvEpiPair {
  float y0, y1;
  float4 e;
  bool rotated;
  __device__ __forceinline__ void load(const Dims& d, const float2* rope, const float* bias, uint32_t pos,
                                       uint32_t hb, uint32_t i, const float* __restrict__ y) {
    const uint32_t r0 = hb * d.hd + i;
    y0 = y[r0];
    y1 = y[r0 + d.half];
    e = make_float4(1.0f, 0.0f, 0.0f, 0.0f);
    rotated = hb < d.nh + d.nkv;
    if (rotated) {
      const float2 cs = rope[(size_t)pos * d.half + i];
      e.x = cs.x;
      e.y = cs.y;
    }
    if (bias) {
      e.z = bias[r0];
      e.w = bias[r0 + d.half];
    }
  }
  __device__ __forceinline__ float2 value(float iv) const {
    const float z0 = y0 * iv + e.z, z1 = y1 * iv + e.w;
    if (!rotated) return make_float2(z0, z1);
    return make_float2(z0 * e.x - z1 * e.y, z1 * e.x + z0 * e.y);
  }
};

// k (hb < nh + nkv) or v rows of head block hb into the row's cache at its
// position (model.rs:466-467).
__device__ __forceinline__ void qkv_epi_cache(const Dims& d, const BRow& r, uint32_t l, uint32_t hb,
                                              uint32_t i, float2 v) {
  const bool is_k = hb < d.nh + d.nkv;
  const uint32_t gi = is_k ? hb - d.nh : hb - d.nh - d.nkv;
  float* row = (is_k ? r.kc : r.vc) + (((size_t)l * d.nkv + gi) * r.cap + r.pos) * d.kvs;
  row[i] = v.x;
  row[i + d.half] = v.y;
}

// QKV epilogue per (row, pair) for the attention items of rows that do not
// run as tiles: q/k/v words tagged; k, v into the row's cache at its position.
__global__ void k_b_qkv_epi(const Args* __restrict__ ap, const BRow* __restrict__ rows, uint32_t l,
                            const float* __restrict__ Y, uint32_t ldy, const float* __restrict__ inv,
                            u64* __restrict__ qkvt, uint32_t ldq) {
  const Dims& d = ap->d;
  const uint32_t b = blockIdx.y;
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= d.qkv_rows / 2) return;
  const BRow r = rows[b];
  const uint32_t hb = p / d.half, i = p - hb * d.half;
  const uint32_t r0 = hb * d.hd + i, r1 = r0 + d.half;
  QkvEpiPair ep;
  ep.load(d, ap->rope, ap->layers[l].bqkv, r.pos, hb, i, Y + (size_t)b * ldy);
  const float2 v = ep.value(inv[b]);
  const u64 g = (u64)gen_of(d, r.tick, l, PH_QKV) << 32;
  qkvt[(size_t)b * ldq + r0] = g | __float_as_uint(v.x);
  qkvt[(size_t)b * ldq + r1] = g | __float_as_uint(v.y);
  if (hb >= d.nh) qkv_epi_cache(d, r, l, hb, i, v);
}

// LDS of the batched kernels that run one-token functions: no weight
// staging (lds_stg = 0 in the row Args).
__device__ __forceinline__ Lds lds_init_rows(const Dims& d) {
  extern __shared__ float lds_raw[];
  Lds s = lds_layout(lds_raw, d);
  if (threadIdx.x == 0) s.ctl->abort_seen = 0;
  __syncthreads();
  return s;
}

// LDS of the attention-only workgroups: the wait control words, then the
// attention's scratch.
__device__ __forceinline__ Lds lds_init_attn() {
  extern __shared__ float lds_raw[];
  Lds s;
  s.ctl = reinterpret_cast<WaitCtl*>(lds_raw);
  s.red = lds_raw + 4;
  s.vec = s.vec2 = s.stg = nullptr;
  s.scr = lds_raw + 4 + 64;
  s.pub = nullptr;
  if (threadIdx.x == 0) s.ctl->abort_seen = 0;
  __syncthreads();
  return s;
}

// Attention items of every row, one per workgroup: entry x of `items` is
// (row, item) packed as row << 16 | item, and the workgroup runs that item
// with the one-token path's phase_attn in its grouped form (item = (kv head,
// chunk) with all the group's query heads; each head's arithmetic is the
// one-token path's), reading the row's tagged q/k/v and writing its tagged
// partials. The workgroups are the NCW attention waves alone (they also
// poll and publish) with only the attention's LDS, so that several items
// share a CU: one row's chunk is a chain of dependent loads and barriers
// that a lone workgroup cannot keep the CU busy with. One score pass and
// four value steps in flight per lane keep the kernel within 128 VGPRs,
// four workgroups per CU.
__global__ __launch_bounds__(NCW * WAVE) __attribute__((amdgpu_waves_per_eu(4))) void k_b_attn_w(
    const Args* __restrict__ rargs, const BRow* __restrict__ rows,
    const uint32_t* __restrict__ items, uint32_t l) {
  const uint32_t e = items[blockIdx.x], b = e >> 16, x = e & 0xffffu;
  const Args& a = rargs[b];
  const Lds s = lds_init_attn();
  const BRow r = rows[b];
  phase_attn<true, 0, NCW, 1, 4>(a, l, r.tick, r.pos, x, 0x10000u, s);
}

// Chunk partials between launches: [row][nh][MAX_ACHUNKS][hd + 4] floats, acc
// first, then m and l (16-byte aligned rows).
__host__ __device__ constexpr uint32_t at_part_row(uint32_t hd) { return hd + 4; }

// Attention of rows with distinct caches (a lockstep step), QKV epilogue and
// chunk combine included: one workgroup per (row, kv head), of TEAMS teams of
// NCW waves. The first waves form 1/rms of the row and the group's q/k/v from
// the QKV product (QkvEpiPair; k and v go to the cache too: no chunk reads
// that row, as position pos comes from LDS). The teams take the chunks in
// turn (team t: chunks t, t + TEAMS, ...), each computing its chunk's
// partials as phase_attn's grouped form does -- the same lanes, chains and
// folds per head, with the next chunk's first K and V rows in flight -- into
// LDS, where combine_scales / combine_value then merge them in chunk order
// into the attention panel.
//
// Bound by latency for few rows (a chain of dependent loads and barriers),
// by memory for many. One workgroup per (row, kv head, chunk) instead, the
// last of a group (an agent-scope count) polling the others' partials, took
// 13.7 us per layer for 7 rows of the 135M shape at 150 positions (11.8 now,
// with the rows' 1/rms inside) and 30 us for 64 of the 1B shape at 256 (27.4).
// Few rows with long histories leave most CUs idle that way (two rows of the
// 135M shape at 4,000 positions: 6 workgroups of 16 chunks each). Then a
// group's chunks are dealt to `splits` workgroups, each with the q/k/v of its
// own, and the partials go to part_g for k_b_comb to merge (the same values,
// the same order). A step of two 135M sessions at 4,000 positions takes 1.41 ms
// so, 2.76 with a workgroup each, at 1,000 positions 1.20 and 1.53.
// HD: the head size, or 0 to read it from d.
struct AttnRowsLds {
  uint32_t ml, sc, wp, part, sw, total;  // float offsets: after q, k and v
};
__host__ __device__ inline AttnRowsLds attn_rows_lds(uint32_t hd, uint32_t grp, uint32_t teams,
                                                     uint32_t ch, uint32_t nch) {
  AttnRowsLds o;
  o.ml = (grp + 2) * hd;                         // [teams][grp][2]
  o.sc = o.ml + teams * 2 * MAX_GROUP;           // [teams][grp][ch]
  o.wp = o.sc + teams * grp * ch;                // [teams][NCW][grp][hd]
  o.part = o.wp + teams * NCW * grp * hd;        // [grp][nch][hd + 2]
  o.sw = o.part + grp * nch * (hd + 2);          // [grp][nch] weights, then [grp] totals
  o.total = o.sw + grp * nch + MAX_GROUP;
  return o;
}
template <uint32_t HD, uint32_t TEAMS, bool SPLIT>
__global__ __launch_bounds__(TEAMS * NCW * WAVE) __attribute__((amdgpu_waves_per_eu(4))) void k_b_attn_f(
    const Args* __restrict__ ap, const BRow* __restrict__ rows, uint32_t l,
    const float* __restrict__ X, const float* __restrict__ Y, uint32_t ldy, uint32_t max_nch,
    uint32_t max_ch, float* __restrict__ attp, uint32_t n_splits, float* __restrict__ part_g) {
  extern __shared__ float lds_raw[];
  // K rows of KU score passes and V rows of VE value steps are requested a
  // chunk ahead, V rows up to VU steps once the scores have freed K's registers.
  constexpr uint32_t KU = HD ? 2 : 1, VE = 4, VU = HD == 64 ? 8 : HD ? 6 : 4, NW = TEAMS * NCW;
  const Args& a = *ap;  // by reference: as kernel arguments its fields took registers (spills, 32 against 27 us at 1B)
  const Dims& d = a.d;
  const uint32_t splits = SPLIT ? n_splits : 1, groups = gridDim.x / splits;
  const uint32_t sp = SPLIT ? blockIdx.x / groups : 0, bg = blockIdx.x - sp * groups;
  const uint32_t b = bg / d.nkv, g = bg - b * d.nkv;
  const BRow r = rows[b];
  const uint32_t pos = r.pos, nch = attn_nchunks(pos), CH = attn_chunk(pos);
  if (SPLIT && sp * TEAMS >= nch) return;  // a shorter row: no chunk of its own
  const uint32_t hd = HD ? HD : d.hd, half = hd / 2, grp = d.group, hs = hd + 2;
  const AttnRowsLds o = attn_rows_lds(hd, grp, TEAMS, max_ch, max_nch);
  const uint32_t wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
  const uint32_t team = wave / NCW, aw = wave % NCW, tt = threadIdx.x % (NCW * WAVE);
  float* qs = lds_raw;  // [grp][hd]
  float* kn = qs + grp * hd;
  float* vn = kn + hd;
  float* ml = lds_raw + o.ml + team * 2 * MAX_GROUP;
  float* sc = lds_raw + o.sc + team * grp * max_ch;  // [grp][CH]
  float* wp = lds_raw + o.wp + team * NCW * grp * hd;
  float* part = lds_raw + o.part;
  AttGeo ge = att_geo(hd);
  const uint32_t ps = lane / ge.lps, sub = lane % ge.lps, pl = lane / ge.lv, dl = lane % ge.lv;
  const uint32_t sstep = NCW * ge.pw, vstep = NCW * ge.pv;
  const uint32_t tw = aw * ge.pw + ps, vw = aw * ge.pv + pl;
  // Uniform bases and 32-bit byte offsets: K and V rows of this kv head.
  const float* kb = r.kc + ((size_t)l * d.nkv + g) * r.cap * d.kvs;
  const float* vb = r.vc + ((size_t)l * d.nkv + g) * r.cap * d.kvs;
  auto load_k = [&](float4 (&k)[4], uint32_t t) {
    const uint32_t at = (t * d.kvs + sub * 16) * 4;
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) k[i] = ldg4_at(kb, at + 16 * i);
  };
  auto load_v = [&](uint32_t t) { return ldg4_at(vb, (t * d.kvs + dl * 4) * 4); };
  float4 kr[KU][4], vr[VU];
  // Rows at or past pos are clamped to the last one before it and never
  // used; the loads have no condition (also for a chunk past the last), so
  // no old value is kept alive for them.
  const uint32_t t_last = max(pos, 1u) - 1;
  auto prefetch = [&](uint32_t c) {
    const uint32_t t0 = c * CH;
#pragma unroll
    for (uint32_t u = 0; u < KU; ++u) load_k(kr[u], min(t0 + tw + u * sstep, t_last));
#pragma unroll
    for (uint32_t u = 0; u < VE; ++u) vr[u] = load_v(min(t0 + vw + u * vstep, t_last));
  };
  prefetch(sp * TEAMS + team);
  // q, k and v of the group: one thread per pair of rotated elements.
  const uint32_t pairs = (grp + 2) * half;
  if (wave * WAVE < pairs) {
    const float iv = rms_row_inv(X + (size_t)b * d.h, d.h, d.eps, lane);
    for (uint32_t u = threadIdx.x; u < pairs; u += NW * WAVE) {
      const uint32_t j = u / half, i = u - j * half;
      const uint32_t hb = j < grp ? g * grp + j : (j == grp ? d.nh + g : d.nh + d.nkv + g);
      QkvEpiPair ep;
      ep.load(d, a.rope, a.layers[l].bqkv, pos, hb, i, Y + (size_t)b * ldy);
      const float2 v = ep.value(iv);
      float* dst = qs + j * hd;  // k and v follow the queries
      lds_st(dst + i, v.x);
      lds_st(dst + i + half, v.y);
      if (j >= grp && sp == 0) qkv_epi_cache(d, r, l, hb, i, v);
    }
  }
  __syncthreads();
  for (uint32_t c0 = sp * TEAMS; c0 < nch; c0 += TEAMS * splits) {
    const uint32_t c = c0 + team, t0 = c * CH;
    const uint32_t t1 = c < nch ? min(t0 + CH, pos + 1) : t0;  // an idle team only meets the barriers
    // scores, KU passes per round
    for (uint32_t pb0 = t0; pb0 < t1; pb0 += KU * sstep) {
#pragma unroll
      for (uint32_t u = 0; u < KU; ++u) {
        const uint32_t ts = pb0 + u * sstep + tw;
        if (ts == pos) {
#pragma unroll
          for (uint32_t i = 0; i < 4; ++i) kr[u][i] = lds4(kn + sub * 16 + 4 * i);
        }
#pragma unroll 1
        for (uint32_t j = 0; j < grp; ++j) {
          float acc = 0.0f;
#pragma unroll
          for (uint32_t i = 0; i < 4; ++i) {
            const float4 qq = lds4(qs + j * hd + sub * 16 + 4 * i);
            acc = fmaf(qq.x, kr[u][i].x, acc);
            acc = fmaf(qq.y, kr[u][i].y, acc);
            acc = fmaf(qq.z, kr[u][i].z, acc);
            acc = fmaf(qq.w, kr[u][i].w, acc);
          }
          const float v = group_sum(acc, ge.lps);
          if (ts < t1 && sub == 0) lds_st(sc + j * CH + (ts - t0), v * d.scale);
        }
        const uint32_t tn = ts + KU * sstep;
        if (tn < t1 && tn < pos) load_k(kr[u], tn);
      }
    }
#pragma unroll
    for (uint32_t u = VE; u < VU; ++u) vr[u] = load_v(min(t0 + vw + u * vstep, t_last));
    __syncthreads();
    // softmax statistics, one wave of the team per query head
    const uint32_t n = t1 - t0;
    if (n > 0 && aw < grp) {
      float* sh = sc + aw * CH;
      float m = -INFINITY;
      for (uint32_t i = lane; i < n; i += WAVE) m = fmaxf(m, lds_ld(sh + i));
      m = wave_max(m);
      float ls = 0.0f;
      for (uint32_t i = lane; i < n; i += WAVE) {
        const float e = (m == -INFINITY) ? 0.0f : expf(lds_ld(sh + i) - m);
        lds_st(sh + i, e);
        ls += e;
      }
      ls = wave_sum(ls);
      if (lane == 0) {
        lds_st(ml + 2 * aw, m);
        lds_st(ml + 2 * aw + 1, ls);
      }
    }
    __syncthreads();
    // exp-weighted V rows: positions t0 + vw + k*vstep, k = 0, 1, ...
    float4 acc[MAX_GROUP];
#pragma unroll
    for (uint32_t j = 0; j < MAX_GROUP; ++j) acc[j] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const uint32_t nk = t0 + vw < t1 ? (t1 - t0 - vw + vstep - 1) / vstep : 0;
    for (uint32_t k0 = 0; k0 < nk; k0 += VU) {
#pragma unroll
      for (uint32_t u = 0; u < VU; ++u) {
        const uint32_t k = k0 + u;
        if (k < nk) {
          const uint32_t t = t0 + vw + k * vstep;
          const float4 v = (t == pos) ? lds4(vn + dl * 4) : vr[u];
          const uint32_t tf = t + VU * vstep;
          if (k + VU < nk && tf < pos) vr[u] = load_v(tf);
#pragma unroll
          for (uint32_t j = 0; j < MAX_GROUP; ++j) {
            if (j >= grp) break;
            const float p = lds_ld(sc + j * CH + (t - t0));
            acc[j].x = fmaf(p, v.x, acc[j].x);
            acc[j].y = fmaf(p, v.y, acc[j].y);
            acc[j].z = fmaf(p, v.z, acc[j].z);
            acc[j].w = fmaf(p, v.w, acc[j].w);
          }
        }
      }
    }
    prefetch(c + TEAMS * splits);
    for (uint32_t x = ge.lv; x < WAVE; x <<= 1) {
#pragma unroll
      for (uint32_t j = 0; j < MAX_GROUP; ++j) {
        if (j >= grp) break;
        acc[j].x += __shfl_xor(acc[j].x, x);
        acc[j].y += __shfl_xor(acc[j].y, x);
        acc[j].z += __shfl_xor(acc[j].z, x);
        acc[j].w += __shfl_xor(acc[j].w, x);
      }
    }
#pragma unroll
    for (uint32_t j = 0; j < MAX_GROUP; ++j)
      if (j < grp && pl == 0) {
        float* dst = wp + (aw * grp + j) * hd + dl * 4;
        lds_st(dst + 0, acc[j].x);
        lds_st(dst + 1, acc[j].y);
        lds_st(dst + 2, acc[j].z);
        lds_st(dst + 3, acc[j].w);
      }
    __syncthreads();
    // The four waves' sums, in wave order, and (m, l). The next round's
    // barriers order these reads before its writes of wp and ml.
    if (n > 0)
      for (uint32_t u = tt; u < grp * hd; u += NCW * WAVE) {
        const uint32_t j = u / hd, dd = u - j * hd;
        float A = 0.0f;
#pragma unroll
        for (uint32_t w = 0; w < NCW; ++w) A += lds_ld(wp + (w * grp + j) * hd + dd);
        if (SPLIT) {  // the tiled attention's layout of the partials
          float* out = part_g + (((size_t)b * d.nh + g * grp + j) * MAX_ACHUNKS + c) * at_part_row(hd);
          out[dd] = A;
          if (dd == 0) {
            out[hd] = lds_ld(ml + 2 * j);
            out[hd + 1] = lds_ld(ml + 2 * j + 1);
          }
          continue;
        }
        float* out = part + (j * nch + c) * hs;
        lds_st(out + 2 + dd, A);
        if (dd == 0) {
          lds_st(out, lds_ld(ml + 2 * j));
          lds_st(out + 1, lds_ld(ml + 2 * j + 1));
        }
      }
  }
  if (SPLIT) return;
  __syncthreads();
  float* sw = lds_raw + o.sw;         // [grp][nch]
  float* ls = sw + grp * max_nch;     // [grp]
  if (threadIdx.x < grp) {
    const float* pj = part + threadIdx.x * nch * hs;
    ls[threadIdx.x] = combine_scales([&](uint32_t i) { return lds_ld(pj + i); }, nch, hs, sw + threadIdx.x * nch);
  }
  __syncthreads();
  for (uint32_t v = threadIdx.x; v < grp * hd; v += NW * WAVE) {
    const uint32_t k = v / hd, dd = v - k * hd, u = (g * grp + k) * hd + dd;
    attp[panel_at(b, u, panel_chunks(d.q))] =
        combine_value([&](uint32_t i) { return lds_ld(part + k * nch * hs + i); }, nch, hs, dd,
                      sw + k * nch, ls[k]);
  }
}

// ----------------------------------------------------- tiled attention
//
// Rows of one cache at consecutive positions (a prefill or a replay) share
// their K/V rows, so their attention runs as tiles: a workgroup takes 16
// consecutive query positions (aligned to 16), one chunk of key positions
// (attn_chunk: 128 * NB) and nj query heads of one kv head, and computes
// every query's chunk partials (m, l, acc) in the order phase_attn uses, with
// MFMA chains where phase_attn has fma chains:
//  * score(q, t): HD / 16 chains of 16 elements (the lanes of a position),
//    then their tree, times scale;
//  * softmax: phase_attn's sums -- lane slot L = 0..63 adds positions L,
//    L + 64, ... from +0, then the wave tree over the 64 slots -- with 16
//    lanes per (query, head), lane s holding slots s + 16v, so a wave takes
//    four (query, head) rows at once;
//  * value[d]: NCW * PV position groups (attention wave w, group pl:
//    positions PV*w + pl + NCW*PV*k, k ascending), each a chain, then per w
//    the tree over its PV groups and the sum w = 0..3 in order, from +0.
// Positions past a query's own (t > pos) carry probability +0, and V rows
// past the tile's last position are zeros: both leave an accumulator
// unchanged (a chain started at +0 never holds -0) as long as the V row is
// finite, 0 * inf being NaN. So a wave looks at its rows of the tile's own
// positions, and where one holds an infinity or a NaN it forms its sums
// again, each query's over the positions it sees alone.
//
// K and V rows go from memory (L2: the tiles of a chunk run on one XCD)
// straight into the registers of the one wave that uses them -- wave w takes
// every fourth key tile for the scores and phase_attn's wave-w position
// groups for the values -- so LDS holds only the query operands, the scores
// and one head's partial sums per wave. A lane loads four consecutive
// elements of a K row and the wave transposes them into MFMA operands with
// lane swaps. Staging K and V in LDS instead (64 KB per task, two workgroups
// per CU, half the clocks in LDS stores and loads) took 100 us per layer for
// 2048 rows of the 135M shape and could not take chunks past 128 positions
// or head_dim 128.

constexpr uint32_t AT_MAX_NB = 4;  // chunks of up to 512 positions (8192 cached)
__host__ __device__ constexpr uint32_t at_pitch(uint32_t ch) { return ch + 17; }  // floats of a score row
// LDS of a task of nj heads: the query operands (then one head's partial
// sums per wave), the score rows, (m, l) per row.
__host__ __device__ constexpr uint32_t attn_tile_lds(uint32_t hd, uint32_t nb, uint32_t nj) {
  const uint32_t qo = nj * hd * 16, wx = NCW * 16 * hd;
  return 4 * ((qo > wx ? qo : wx) + nj * 16 * (at_pitch(nb * ACHUNK) + 2));
}
// v[0..3] of lane (lr, lc) = elements 4*lc .. 4*lc+3 of row lr; afterwards
// v[i] = element 4*i + lc (a 4x4 transpose between components and the wave's
// four rows of 16 lanes).
__device__ __forceinline__ void transpose4(float4& v) {
  auto swap32 = [](float& a, float& b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(r[0]);
    b = __uint_as_float(r[1]);
  };
  auto swap16 = [](float& a, float& b) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(r[0]);
    b = __uint_as_float(r[1]);
  };
  swap32(v.x, v.z);
  swap32(v.y, v.w);
  swap16(v.x, v.y);
  swap16(v.z, v.w);
}

// The complete tree over N chain sums (N = 4 or 8).
template <int N>
__device__ __forceinline__ f4v chain_tree(const f4v (&a)[N]) {
  const f4v t = (a[0] + a[1]) + (a[2] + a[3]);
  if constexpr (N == 8) return t + ((a[4] + a[5]) + (a[6] + a[7]));
  return t;
}

// tasks[x] = tile << 16 | chunk << 8 | kv head, each run ny times for nj
// query heads (heads y*nj ..); tiles[m] .. tiles[m + 1] are the batch rows of
// tile m. rows: the batch (one cache, consecutive positions); qf: the rows'
// rotated queries [row][q]; part: the chunk partials.
template <int HD, int NB>
__global__ __launch_bounds__(256, 2) void k_b_attn_tile(const Dims d, const BRow* __restrict__ rows,
                                                     const uint32_t* __restrict__ tasks, uint32_t ny,
                                                     uint32_t nj, const uint32_t* __restrict__ tiles,
                                                     uint32_t l, const float* __restrict__ qf,
                                                     float* __restrict__ part) {
  constexpr int SUBS = HD / 16;                  // chains of a score
  constexpr int PV = WAVE / (HD / 4);            // value position groups of a wave (phase_attn's pv)
  constexpr int GV = NCW * PV;                   // ... of all waves: a group's positions are GV apart
  constexpr int HH = HD / 64;                    // 64-dim halves of a V row
  constexpr uint32_t CH = NB * ACHUNK, SP = at_pitch(CH);
  constexpr int MB = ACHUNK / (4 * GV);          // value MFMA steps of 128 positions
  constexpr bool HOLD = NB * HD <= 128;          // a chunk's V rows fit the registers for all heads
  extern __shared__ float at_lds[];
  const uint32_t tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE;
  const uint32_t lr = lane % 16, lc = lane / 16;
  // Consecutive tasks (same chunk and kv head, the next tile) on one XCD.
  const uint32_t n_wg = gridDim.x, xk = blockIdx.x % NXCD;
  const uint32_t ti = xk * (n_wg / NXCD) + min(xk, n_wg % NXCD) + blockIdx.x / NXCD;
  const uint32_t task = tasks[ti / ny], j0 = ti % ny * nj, njt = min(nj, d.group - j0);
  const uint32_t m = task >> 16, c = (task >> 8) & 0xffu, g = task & 0xffu;
  const uint32_t rb0 = tiles[m], nq = tiles[m + 1] - rb0;
  const BRow r0 = rows[rb0];
  const uint32_t p_last = r0.pos + nq - 1, t0 = c * CH;
  const uint32_t nk = min(CH, p_last + 1 - t0);
  const uint32_t qo_n = nj * HD * 16, wx_n = NCW * 16 * HD;
  float* Qo = at_lds;                                  // [nj][SUBS][lane][4]: MFMA operands
  float* Wx = at_lds;                                  // [NCW][16][HD], once the scores are done
  float* Ss = at_lds + (qo_n > wx_n ? qo_n : wx_n);    // [nj][16][SP]: scores, then probabilities
  float* ML = Ss + nj * 16 * SP;                       // [nj][16][2]: m, l
  const float* kb = r0.kc + ((size_t)l * d.nkv + g) * r0.cap * HD;
  const float* vb = r0.vc + ((size_t)l * d.nkv + g) * r0.cap * HD;
  // 1. Query operands: wave w prepares every fourth (head, chain).
  const float* qrow = qf + (size_t)(rb0 + min(lr, nq - 1)) * d.q + (size_t)(g * d.group + j0) * HD + 4 * lc;
  for (uint32_t u = wave; u < njt * SUBS; u += NCW) {
    float4 v = ldg4(qrow + 16 * u);  // chains of consecutive heads are 16 elements apart
    transpose4(v);
    *reinterpret_cast<float4*>(Qo + (size_t)(u * WAVE + lane) * 4) = v;
  }
  // The wave's first key tile is requested before the barrier.
  const uint32_t nkt = (nk + 15) / 16;
  float4 kf[SUBS];
  auto load_k = [&](uint32_t kt) {
    const float* r = kb + (size_t)min(t0 + kt * 16 + lr, p_last) * HD + 4 * lc;
#pragma unroll
    for (int u = 0; u < SUBS; ++u) kf[u] = ldg4(r + 16 * u);
  };
  if (wave < nkt) load_k(wave);
  __syncthreads();
  // 2. Scores of the wave's key tiles, the next tile's rows in flight.
#pragma unroll 1
  for (uint32_t kt = wave; kt < nkt; kt += NCW) {
    float4 ka[SUBS];
#pragma unroll
    for (int u = 0; u < SUBS; ++u) {
      ka[u] = kf[u];
      transpose4(ka[u]);
    }
    if (kt + NCW < nkt) load_k(kt + NCW);
#pragma unroll 1
    for (uint32_t j = 0; j < njt; ++j) {
      float4 qa[SUBS];
#pragma unroll
      for (int u = 0; u < SUBS; ++u)
        qa[u] = *reinterpret_cast<const float4*>(Qo + (size_t)((j * SUBS + u) * WAVE + lane) * 4);
      f4v acc[SUBS];
#pragma unroll
      for (int u = 0; u < SUBS; ++u) acc[u] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int u = 0; u < SUBS; ++u)
          acc[u] = __builtin_amdgcn_mfma_f32_16x16x4f32((&qa[u].x)[i], (&ka[u].x)[i], acc[u], 0, 0, 0);
      const f4v sc = chain_tree(acc);
#pragma unroll
      for (int rr = 0; rr < 4; ++rr)  // query 4*lc + rr, key kt*16 + lr
        Ss[(j * 16 + 4 * lc + rr) * SP + kt * 16 + lr] = sc[rr] * d.scale;
    }
  }
  // The value rows of a 128-position block: wave w's groups PV*w + pl, group
  // positions 4*mm + lc, dims 64*hh + 4*lr .. +3.
  float4 vf[HOLD ? NB : 1][PV][MB][HH];
  auto load_v = [&](int nb, float4 (&v)[PV][MB][HH]) {
#pragma unroll
    for (int pl = 0; pl < PV; ++pl)
#pragma unroll
      for (int mm = 0; mm < MB; ++mm) {
        const uint32_t p = nb * ACHUNK + PV * wave + pl + GV * (4 * mm + lc);
        const float* r = vb + (size_t)min(t0 + p, p_last) * HD + 4 * lr;
#pragma unroll
        for (int hh = 0; hh < HH; ++hh) v[pl][mm][hh] = ldg4(r + 64 * hh);
      }
  };
  auto zero_v = [&](int nb, float4 (&v)[PV][MB][HH]) {  // rows past the tile's last position
    if (nk == CH) return;
#pragma unroll
    for (int pl = 0; pl < PV; ++pl)
#pragma unroll
      for (int mm = 0; mm < MB; ++mm)
        if (nb * ACHUNK + PV * wave + pl + GV * (4 * mm + lc) >= nk)
#pragma unroll
          for (int hh = 0; hh < HH; ++hh) v[pl][mm][hh] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  };
  if constexpr (HOLD)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) load_v(nb, vf[nb]);
  // The wave's V rows at positions that the tile's first query does not see
  // (t > its own): x * 0 is NaN for an infinity or a NaN, +-0 else. The tile's
  // positions lie in one 16-aligned block, four of them the wave's: one per lc.
  const uint32_t p_own = r0.pos - t0;  // past the chunk in all but the tile's last chunk
  float unseen = 0.0f;
  if (p_own < CH) {
    const uint32_t p = p_own / 16 * 16 + PV * wave + lc % PV + GV * (lc / PV);
    if (p > p_own && p < nk) {
      const float* r = vb + (size_t)(t0 + p) * HD + 4 * lr;
#pragma unroll
      for (int hh = 0; hh < HH; ++hh) {
        const float4 x = ldg4(r + 64 * hh);
        unseen += (x.x * 0.0f + x.y * 0.0f) + (x.z * 0.0f + x.w * 0.0f);
      }
    }
  }
  const bool odd = __any(unseen != unseen);
  __syncthreads();
  // 3. Softmax statistics and probabilities, 16 lanes per (query, head):
  // lane sub holds phase_attn's lane slots L = sub + 16v (v = 0..3); the
  // slots' tree is group_sum over the 16 lanes of each v, then (R3 + R2) +
  // (R1 + R0) as wave_sum. Positions from n on get probability +0.
  for (uint32_t u0 = 4 * wave; u0 < njt * 16; u0 += 16) {
    const uint32_t u = u0 + lane / 16, q = u % 16, sub = lane % 16;
    float* sh = Ss + u * SP;
    const uint32_t n = q < nq ? min(CH, r0.pos + q + 1 - t0) : 0;
    float e[8 * NB];
    float mx = -INFINITY;
#pragma unroll
    for (int k = 0; k < 8 * NB; ++k) {
      const uint32_t i = sub + 16 * k;
      e[k] = i < n ? sh[i] : -INFINITY;
      mx = fmaxf(mx, e[k]);
    }
    mx = row_max(mx);
#pragma unroll
    for (int k = 0; k < 8 * NB; ++k) {
      const uint32_t i = sub + 16 * k;
      e[k] = (i < n && mx != -INFINITY) ? expf(e[k] - mx) : 0.0f;
      sh[i] = e[k];
    }
    float R[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      float t = 0.0f;
#pragma unroll
      for (int k = 0; k < 2 * NB; ++k) t = t + e[v + 4 * k];
      R[v] = group_sum(t, 16);
    }
    if (sub == 0) {
      ML[u * 2] = mx;
      ML[u * 2 + 1] = (R[3] + R[2]) + (R[1] + R[0]);
    }
  }
  if constexpr (HOLD)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) zero_v(nb, vf[nb]);
  // 4. Values, one head at a time.
#pragma unroll 1
  for (uint32_t j = 0; j < njt; ++j) {
    f4v acc[PV][HH][4];
#pragma unroll
    for (int pl = 0; pl < PV; ++pl)
#pragma unroll
      for (int hh = 0; hh < HH; ++hh)
#pragma unroll
        for (int u = 0; u < 4; ++u) acc[pl][hh][u] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (!HOLD) load_v(0, vf[0]);
    __syncthreads();  // the probabilities (j = 0), or the last head's Wx read, are done
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      if constexpr (!HOLD) {
        if (nb > 0) load_v(nb, vf[0]);
        zero_v(nb, vf[0]);
      }
      float4 (&v)[PV][MB][HH] = vf[HOLD ? nb : 0];
#pragma unroll
      for (int mm = 0; mm < MB; ++mm)
#pragma unroll
        for (int pl = 0; pl < PV; ++pl) {
          const float p = Ss[(j * 16 + lr) * SP + nb * ACHUNK + PV * wave + pl + GV * (4 * mm + lc)];
#pragma unroll
          for (int hh = 0; hh < HH; ++hh)
#pragma unroll
            for (int u = 0; u < 4; ++u)
              acc[pl][hh][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(p, (&v[pl][mm][hh].x)[u],
                                                                    acc[pl][hh][u], 0, 0, 0);
        }
    }
#pragma unroll
    for (int hh = 0; hh < HH; ++hh) {
      f4v w[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        w[u] = acc[0][hh][u] + acc[1][hh][u];
        if constexpr (PV == 4) w[u] = w[u] + (acc[2][hh][u] + acc[3][hh][u]);
      }
#pragma unroll
      for (int rr = 0; rr < 4; ++rr)  // query 4*lc + rr, dims 64*hh + 4*lr ..
        *reinterpret_cast<float4*>(Wx + (size_t)(wave * 16 + 4 * lc + rr) * HD + 64 * hh + 4 * lr) =
            make_float4(w[0][rr], w[1][rr], w[2][rr], w[3][rr]);
    }
    if (odd) {  // wave-uniform
#pragma unroll 1
      for (uint32_t q = 0; q < nq; ++q)
#pragma unroll 1
        for (uint32_t dd = lane; dd < HD; dd += WAVE) {
          float g4[PV];
#pragma unroll
          for (int pl = 0; pl < PV; ++pl) {
            g4[pl] = 0.0f;
#pragma unroll 1
            for (uint32_t p = PV * wave + pl; p < nk && p <= p_own + q; p += GV)
              g4[pl] = fmaf(Ss[(j * 16 + q) * SP + p], vb[(size_t)(t0 + p) * HD + dd], g4[pl]);
          }
          float A = g4[0] + g4[1];
          if constexpr (PV == 4) A = A + (g4[2] + g4[3]);
          Wx[(size_t)(wave * 16 + q) * HD + dd] = A;
        }
    }
    __syncthreads();
    const uint32_t hidx = g * d.group + j0 + j;
#pragma unroll
    for (uint32_t e = tid * 4; e < 16 * HD; e += 1024) {
      const uint32_t q = e / HD, dd = e % HD;
      float4 A = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
      for (uint32_t w = 0; w < NCW; ++w) {
        const float4 x = *reinterpret_cast<const float4*>(Wx + (size_t)w * 16 * HD + e);
        A = make_float4(A.x + x.x, A.y + x.y, A.z + x.z, A.w + x.w);
      }
      if (q >= nq) continue;
      float* out = part + (((size_t)(rb0 + q) * d.nh + hidx) * MAX_ACHUNKS + c) * at_part_row(HD);
      *reinterpret_cast<float4*>(out + dd) = A;
      if (dd == 0) {
        out[HD] = ML[(j * 16 + q) * 2];
        out[HD + 1] = ML[(j * 16 + q) * 2 + 1];
      }
    }
  }
}

// Combine of the chunk partials (combine_scales / combine_value, as the O
// phase does) into the panel of att[b][q]: one workgroup per row and group of
// heads; the weights of a head's chunks are formed once in LDS (a wave per
// head, a lane per chunk), then a thread per (head, dim). The partials were
// written by earlier launches on the same stream, so their values are read
// directly: TILED, the tiled attention's floats; otherwise the low half of
// each tagged word (m, l, acc).
constexpr uint32_t COMB_MAX_HEADS = 64;
constexpr uint32_t COMB_HEADS_PER_BLOCK = 4;  // grid y: groups of heads
template <bool TILED>
__global__ __launch_bounds__(256) void k_b_comb(const Dims d, const BRow* __restrict__ rows,
                                                const u64* __restrict__ part, uint32_t part_w,
                                                float* __restrict__ attp) {
  __shared__ float sc[COMB_HEADS_PER_BLOCK][MAX_ACHUNKS];
  __shared__ float ls[COMB_HEADS_PER_BLOCK];
  const uint32_t b = blockIdx.x, h0 = blockIdx.y * COMB_HEADS_PER_BLOCK;
  const uint32_t nh = min(COMB_HEADS_PER_BLOCK, d.nh - h0);
  const uint32_t nch = attn_nchunks(rows[b].pos);
  // Float i (0: m, 1: l, 2 + dim: acc) of chunk c of head h0 + k.
  const u64* pb = part + (size_t)b * part_w;
  const float* pf = reinterpret_cast<const float*>(part) + (size_t)b * d.nh * MAX_ACHUNKS * at_part_row(d.hd);
  auto val = [&](uint32_t k, uint32_t c, uint32_t i) {
    const size_t at = (size_t)(h0 + k) * MAX_ACHUNKS + c;
    if (TILED) return pf[at * at_part_row(d.hd) + (i < 2 ? d.hd + i : i - 2)];
    return __uint_as_float((uint32_t)pb[at * (d.hd + 2) + i]);
  };
  const uint32_t wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
  // combine_scales for head h0 + wave, one lane per chunk: M is a maximum
  // (the same in any order, NaN maxima dropped as fmaxf from -inf drops
  // them), each weight the same expf, and the weighted total summed in
  // chunk order by lane 0 from the lanes' products (no contraction).
  if (wave < nh) {
    if (nch == 1) {
      if (lane == 0) ls[wave] = val(wave, 0, 1) * 1.0f;
    } else {
      const float mc = lane < nch ? val(wave, lane, 0) : -INFINITY;
      const float lc = lane < nch ? val(wave, lane, 1) : 0.0f;
      float M = fmaxf(-INFINITY, mc);
      for (int o = 32; o > 0; o >>= 1) M = fmaxf(M, __shfl_xor(M, o));
      const float w = (mc == -INFINITY) ? 0.0f : expf(mc - M);
      const float prod = lc * w;
      if (lane < nch) sc[wave][lane] = w;
      float Ls = 0.0f;
      for (uint32_t c = 0; c < nch; ++c) Ls = Ls + __shfl(prod, c);
      if (lane == 0) ls[wave] = Ls;
    }
  }
  __syncthreads();
  // combine_value, with the chunks' values loaded before the sum (the same
  // sum in chunk order).
  for (uint32_t v = threadIdx.x; v < nh * d.hd; v += blockDim.x) {
    const uint32_t k = v / d.hd, dd = v - k * d.hd, u = (h0 + k) * d.hd + dd;
    float x[MAX_ACHUNKS];
#pragma unroll
    for (uint32_t c = 0; c < MAX_ACHUNKS; ++c) x[c] = c < nch ? val(k, c, 2 + dd) : 0.0f;
    float out;
    if (nch == 1) {
      out = (x[0] * 1.0f) / ls[k];
    } else {
      float A = 0.0f;
#pragma unroll
      for (uint32_t c = 0; c < MAX_ACHUNKS; ++c)
        if (c < nch) A = A + x[c] * sc[k][c];
      out = A / ls[k];
    }
    attp[panel_at(b, u, panel_chunks(d.q))] = out;
  }
}

// g = act(gate * inv) * (up * inv) (phase_gu), into the panel GP, where the
// product cannot do it itself (GO_ACT: whole 16-row tiles of gate rows); Y holds gate rows then up rows.
__global__ void k_b_act(const float* __restrict__ Y, uint32_t ldy, const float* __restrict__ inv,
                        uint32_t ff, uint32_t act, float* __restrict__ GP) {
  const uint32_t b = blockIdx.y;
  const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= ff) return;
  const float iv = inv[b];
  const float gate = Y[(size_t)b * ldy + j], up = Y[(size_t)b * ldy + ff + j];
  GP[panel_at(b, j, panel_chunks(ff))] = act_fn(gate * iv, act) * (up * iv);
}

// Final norm of the rows that need logits (phase_lm): xs = x * w_norm and
// inv = 1/rms(x) in rms_inv's order; xs goes into the panel XSP. One wave
// per logits row; sel[i] is its batch row.
__global__ __launch_bounds__(64) void k_b_final(const float* __restrict__ X,
                                                const uint32_t* __restrict__ sel, uint32_t h,
                                                const float* __restrict__ nrm, float eps,
                                                float* __restrict__ XSP, float* __restrict__ linv) {
  const uint32_t i = blockIdx.x, lane = threadIdx.x, nch = panel_chunks(h);
  const float* x = X + (size_t)sel[i] * h;
  float ss = 0.0f;
  for (uint32_t j = lane * 4; j < h; j += 256) {
    const float4 v = *reinterpret_cast<const float4*>(x + j);
    ss = fmaf(v.x, v.x, ss);
    ss = fmaf(v.y, v.y, ss);
    ss = fmaf(v.z, v.z, ss);
    ss = fmaf(v.w, v.w, ss);
    XSP[panel_at(i, j, nch)] = v.x * nrm[j];
    XSP[panel_at(i, j + 1, nch)] = v.y * nrm[j + 1];
    XSP[panel_at(i, j + 2, nch)] = v.z * nrm[j + 2];
    XSP[panel_at(i, j + 3, nch)] = v.w * nrm[j + 3];
  }
  ss = wave_sum(ss);
  if (lane == 0) linv[i] = 1.0f / sqrtf(ss / (float)h + eps);
}

// Chunk (max, argmax) of the tagged logits of every logits row, tagged for the
// sampler: each wave takes CM_CPW consecutive chunks, one lane per row of a
// chunk, with all its loads issued before the first reduction (phase_lm's
// reduction; argmax is a total order, so any tree gives its answer).
constexpr uint32_t CM_CPW = 4;
__global__ __launch_bounds__(256) void k_b_chunkmax(const Dims d, const u64* __restrict__ logt,
                                                    const uint32_t* __restrict__ gen,
                                                    u64* __restrict__ vmax, u64* __restrict__ varg,
                                                    uint32_t nlm) {
  const uint32_t c0 = (blockIdx.x * 4 + threadIdx.x / WAVE) * CM_CPW, lane = threadIdx.x % WAVE;
  const uint32_t i = blockIdx.y;
  if (c0 >= d.nvc || i >= nlm) return;
  u64 raw[CM_CPW];
#pragma unroll
  for (uint32_t u = 0; u < CM_CPW; ++u) {
    const uint32_t v = (c0 + u) * VCHUNK + lane;
    raw[u] = (c0 + u < d.nvc && v < d.V) ? logt[(size_t)i * d.V + v] : 0;
  }
  const u64 g = (u64)gen[i] << 32;
#pragma unroll
  for (uint32_t u = 0; u < CM_CPW; ++u) {
    const uint32_t c = c0 + u;
    if (c >= d.nvc) break;
    const uint32_t v = c * VCHUNK + lane;
    float bv = -INFINITY;
    uint32_t bi = NO_INDEX;
    if (v < d.V) {
      const float y = __uint_as_float((uint32_t)raw[u]);
      if (!isnan(y)) {
        bv = y;
        bi = v;
      }
    }
    for (int o = 32; o > 0; o >>= 1) {
      const float v2 = __shfl_xor(bv, o);
      const uint32_t i2 = __shfl_xor(bi, o);
      if (better(v2, i2, bv, bi)) {
        bv = v2;
        bi = i2;
      }
    }
    if (lane == 0) {
      vmax[(size_t)i * d.nvc + c] = g | __float_as_uint(bv);
      varg[(size_t)i * d.nvc + c] = g | bi;
    }
  }
}

// Chunks per wave and round of k_b_sample's stage A: a lone workgroup of an
// op walks all the row's chunks, so rounds of NWA chunks would each wait a
// full memory latency. Its LDS holds NWA * SAMP_CPW chunks past the rows
// layout's scratch start (samp_lds_bytes).
constexpr uint32_t SAMP_CPW = 8;

// Sampling ops, G workgroups each (the one-token sampler, its stages shared
// among them as among the persistent kernel's workgroups): op j samples
// logits row lrow[j] for generation base tick[j] with rng word words[j]; the
// token goes to out[j]. With G > 1 an op's workgroups wait for each other's
// words, so all of them must be resident (a cooperative launch). An op on one
// workgroup is bound by that CU's arithmetic (the exp of every logit) and
// reads: 7 ops of 49,152 logits took 262 us on one workgroup each, 73 on 36.
__global__ __launch_bounds__(BLOCK) void k_b_sample(const Args* __restrict__ largs,
                                                    const uint32_t* __restrict__ tick,
                                                    const uint32_t* __restrict__ words, float T,
                                                    uint32_t tag0, uint32_t G,
                                                    uint32_t* __restrict__ out) {
  const uint32_t j = blockIdx.x / G, wg = blockIdx.x - j * G;
  const Args& a = largs[j];
  const Lds s = lds_init_rows(a.d);
  // A row whose wait runs out still leaves a token in range (0), so a
  // following batched embedding never reads outside the table.
  if (wg == 0 && threadIdx.x == 0) out[j] = 0u;
  uint32_t tok = 0;
  if (T != 0.0f) {
    float m;
    uint32_t bi;
    if (!sample_stage_a<SAMP_CPW, 8>(a, tick[j], tag0 + j, T, wg, G, s, &m, &bi)) return;
    if (!sample_exact(a, tag0 + j, m, bi, words[j], wg, G, true, s, &tok)) return;
  } else if (!sample_greedy(a, tick[j], s, &tok)) {
    return;
  }
  if (wg == 0 && threadIdx.x == 0) out[j] = tok;
}

}  // namespace dg
