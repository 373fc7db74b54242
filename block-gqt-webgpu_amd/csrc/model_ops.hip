// The model step's separate attention passes, by the reference's dispatch
// names (src/model/ops.ts:6-12): append (src/model/append.wgsl:6-10), dot,
// softmax and weighted (src/model/attention.wgsl:13-39) and compressed_dot
// (src/model/compressed-dot.wgsl:14-31). They keep the reference's buffer
// layouts, including the materialised scores and probabilities
// [rows*qHeads, tokens]; the fused decode and prefill kernels are the fast
// path for the same step. Each pass covers the work items the reference's
// dispatch of x (and y) workgroups covers, clamped to the parameters' extents.
#include <hip/hip_fp16.h>

#include "bgtq_internal.h"
#include "gfx950_common.h"

namespace bgtq {
namespace {

using namespace gfx;

__device__ __forceinline__ float h2f(uint16_t h) { return __half2float(__ushort_as_half(h)); }
__device__ __forceinline__ uint16_t f2h(float v) { return __half_as_ushort(__float2half_rn(v)); }

// append.wgsl:6-10: pair i of the rows x heads x 32 pairs (64 dims) of the
// FP32 input, rounded to FP16, into cache[head][start + row][pair].
__global__ __launch_bounds__(256) void model_append_kernel(ModelAppendParams p) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= p.pairs) return;
  const int64_t per_row = (int64_t)p.heads * 32;
  const int64_t row = i / per_row;
  const int head = (int)((i / 32) % p.heads), pair = (int)(i % 32);
  const int64_t at = ((int64_t)head * p.capacity + p.start + row) * 32 + pair;
  const float2 v = reinterpret_cast<const float2 *>(p.input)[i];
  p.cache[at] = (uint32_t)f2h(v.x) | ((uint32_t)f2h(v.y) << 16);
}

// One 16x16x4 FP32 matrix-core product: lane (gq, col) = (lane / 16, lane % 16)
// holds A[col][gq] and B[gq][col]; element r of the result is D[4 gq + r][col].
__device__ __forceinline__ f32x4 mfma_f32(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Scores of the dispatch's query rows against the tokens of one KV head per
// grid z (compressed-dot.wgsl:14-31 with packed K, attention.wgsl:13-23 with
// FP16 K rows). The packed-K dot uses the rotated query:
// q . (R^T c)[perm^-1] = sum_j c_j (R q_perm)_j, with
// c_j = centroid(code_j) * scale(group of j) as the reference forms it.
//
// The pass is a [tokens x d] x [d x query items] product, in FP32 on the
// matrix cores (16x16x4: the scores the reference keeps are FP32, and its
// rate is twice the vector ALUs'). Bound: the latency of one dependent chain
// (codes and queries, the rotation through LDS, the products), not bytes: a
// workgroup is four waves of 32 tokens by 32 query items (row-major rows x
// gqa), so a chunk of 32 rows x 3 heads rebuilds each token's K three times
// instead of 32 and one new token's 4097 scores spread over 33 workgroups a
// head. Lane (gq, col) owns dims 16 n + 4 gq + r of its token and its query:
// the rotation's result (rows 4 gq + r of tile n) then has the operand's
// order. Codes are byte loads (rows have any length and alignment).
// One new token against 4097 of three heads: 7.1 us in one launch (a thread
// per token, one launch per head: 36 us each); 32 rows x 2048 tokens: 12.0 us
// (35 us per head).
// Grid: (token blocks of 128, groups of 32 query items, KV heads).
constexpr int kScoreTokens = 128, kScoreItems = 32;

template <int D, int KF>
__global__ __launch_bounds__(256) void model_scores_kernel(ModelScoresParams p) {
  constexpr int NT = D / 16, QT = kScoreItems / 16;
  __shared__ __align__(16) float qs[KF ? QT * 16 * (D + 4) : 1];
  __shared__ float scl[KF ? kMaxGroups * kScoreTokens : 1];
  extern __shared__ __align__(16) uint8_t smem[];
  float *books = reinterpret_cast<float *>(smem);
  const int tid = threadIdx.x, lane = tid & 63, gq = lane >> 4, col = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int G = p.gqa, items = p.rows * G, q0 = blockIdx.y * kScoreItems;
  const int kv = KF ? p.jobs[blockIdx.z].head : p.head0 + (int)blockIdx.z;
  const int nqt = min(QT, (items - q0 + 15) / 16);
  const int tb = blockIdx.x * kScoreTokens;
  // Tokens past the last row's causal end are never read (their scores are
  // -inf or not written); the lane re-reads the last one.
  const int t_read = min(p.n_tok, p.start + p.rows);

  // This lane's query of each tile (items past the dispatch's: item 0, not stored).
  const float *qv[QT];
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    const int item = q0 + 16 * qt + col < items ? q0 + 16 * qt + col : 0;
    const int row = item / G;
    qv[qt] = p.q + ((int64_t)row * p.q_heads + kv * G + (item - row * G)) * D;
  }
  float kreg[2][NT][4];
  float qreg[QT][NT][4];
  if (KF == 1) {
    const ModelScoresJob &job = p.jobs[blockIdx.z];
    const DevTables *T = job.tables;
    const int nib = T->nibble_dims, rb = T->row_bytes, ns = T->norm_stride, ng = T->groups, mc = T->max_centroids;
    // The loads go out in one batch (the permutation first: the query
    // elements' addresses need it), without branches between them.
    uint32_t pw[NT], pb[NT], pg[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) pw[n] = *reinterpret_cast<const uint32_t *>(T->perm + 16 * n + 4 * gq);
    // qr^T = R q_perm^T: wave w computes rows 16 n .. 16 n + 15 for n = w, w + 4.
    constexpr int NW = NT / 4;
    const float *R = tables_rot(T);
    f32x4 ra[NW][NT];
#pragma unroll
    for (int k = 0; k < NW; ++k)
#pragma unroll
      for (int m = 0; m < NT; ++m)
        ra[k][m] = *reinterpret_cast<const f32x4 *>(R + (16 * (wave + 4 * k) + col) * D + 16 * m + 4 * gq);
    constexpr int NS = kMaxGroups * kScoreTokens / 256;
    uint16_t sv[NS];
#pragma unroll
    for (int k = 0; k < NS; ++k) {
      const int e = min(tid + 256 * k, ng * kScoreTokens - 1);
      sv[k] = job.norms[(int64_t)min(tb + e % kScoreTokens, t_read - 1) * ns + e / kScoreTokens];
    }
    const float *bg = tables_books(T);
    const int nbf = T->n_books * mc;
    constexpr int NB = 4;  // the first 1024 book entries (the rest below)
    float bv[NB];
#pragma unroll
    for (int k = 0; k < NB; ++k) bv[k] = bg[min(tid + 256 * k, nbf - 1)];
    __builtin_amdgcn_sched_barrier(0);
    float x[QT][NT][4];
#pragma unroll
    for (int qt = 0; qt < QT; ++qt)
#pragma unroll
      for (int m = 0; m < NT; ++m)
#pragma unroll
        for (int i = 0; i < 4; ++i) x[qt][m][i] = qv[qt][(pw[m] >> (8 * i)) & 255u];
    // Code bytes of this lane's positions for its two tokens (a byte past the
    // last token read is a zero).
    uint32_t code[2][NT][4];
    {
      const int n_tok = min(t_read - tb, kScoreTokens);
      const __amdgpu_buffer_rsrc_t rk = rsrc(job.packed + (int64_t)tb * rb, (uint32_t)max(n_tok, 0) * (uint32_t)rb);
      const int row0 = (32 * wave + col) * rb, row1 = row0 + 16 * rb;
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int j = 16 * n + 4 * gq + r, off = j < nib ? j >> 1 : (nib >> 1) + j - nib;
          code[0][n][r] = (uint8_t)__builtin_amdgcn_raw_buffer_load_b8(rk, row0 + off, 0, 0);
          code[1][n][r] = (uint8_t)__builtin_amdgcn_raw_buffer_load_b8(rk, row1 + off, 0, 0);
        }
    }
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      pb[n] = *reinterpret_cast<const uint32_t *>(T->pos_book + 16 * n + 4 * gq);
      pg[n] = *reinterpret_cast<const uint32_t *>(T->group_of + 16 * n + 4 * gq);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < NS; ++k)
      if (tid + 256 * k < ng * kScoreTokens) scl[tid + 256 * k] = h2f(sv[k]);
#pragma unroll
    for (int k = 0; k < NB; ++k)
      if (tid + 256 * k < nbf) books[tid + 256 * k] = bv[k];
    for (int e = tid + 256 * NB; e < nbf; e += 256) books[e] = bg[e];
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      if (qt >= nqt) break;
#pragma unroll
      for (int k = 0; k < NW; ++k) {
        f32x4 acc = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int m = 0; m < NT; ++m)
#pragma unroll
          for (int i = 0; i < 4; ++i) acc = mfma_f32(ra[k][m][i], x[qt][m][i], acc);
        *reinterpret_cast<f32x4 *>(qs + (16 * qt + col) * (D + 4) + 16 * (wave + 4 * k) + 4 * gq) = acc;
      }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int j = 16 * n + 4 * gq + r;
          const uint32_t c = j < nib ? (code[u][n][r] >> ((j & 1) * 4)) & 15u : code[u][n][r];
          const float s = scl[((pg[n] >> (8 * r)) & 255u) * kScoreTokens + 32 * wave + 16 * u + col];
          kreg[u][n][r] = books[((pb[n] >> (8 * r)) & 255u) * mc + c] * s;
        }
#pragma unroll
    for (int qt = 0; qt < QT; ++qt)
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        if (qt >= nqt) break;
        const f32x4 v = *reinterpret_cast<const f32x4 *>(qs + (16 * qt + col) * (D + 4) + 16 * n + 4 * gq);
#pragma unroll
        for (int r = 0; r < 4; ++r) qreg[qt][n][r] = v[r];
      }
  } else {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int t = min(tb + 32 * wave + 16 * u + col, t_read - 1);
      const uint16_t *krow = p.k + ((int64_t)kv * p.capacity + t) * D;
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r) kreg[u][n][r] = h2f(krow[16 * n + 4 * gq + r]);
    }
#pragma unroll
    for (int qt = 0; qt < QT; ++qt)
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r) qreg[qt][n][r] = qt < nqt ? qv[qt][16 * n + 4 * gq + r] : 0.0f;
  }

  // Work item (row, g) of the reference's dispatch: item = row*gqa + g in
  // workgroup row item / 128 (offset by the KV head's blocks for dot).
  const int blocks = (items + 127) / 128;
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    if (qt >= nqt) break;
    const int item = q0 + 16 * qt + col, row = item / G;
    const int wg_row = (KF == 1 ? 0 : (int)blockIdx.z * blocks) + item / 128;
    const bool ok = item < items && wg_row < p.y_limit;
    float *out = p.scores + ((int64_t)row * p.q_heads + kv * G + (item - row * G)) * p.tokens;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      f32x4 acc = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc = mfma_f32(kreg[u][n][r], qreg[qt][n][r], acc);
      const int t0 = tb + 32 * wave + 16 * u + 4 * gq;
#pragma unroll
      for (int r = 0; r < 4; ++r)  // tokens after the row's causal end are -inf
        if (ok && t0 + r < p.n_tok) out[t0 + r] = t0 + r <= p.start + row ? acc[r] * p.scale : -INFINITY;
    }
  }
}

// attention.wgsl:24-31: one workgroup per score row r (= row*qHeads + head):
// probabilities over tokens < end = min(tokens, start + row + 1), zero after.
// A thread keeps up to kRowValues scores (and their exponentials) in
// registers, so a row of up to 8192 tokens is read once and each exponential
// taken once; longer rows go over their tokens again. Bound: one memory round
// trip and two workgroup reductions (9 rows of 4097 tokens: 4.2 us; 12.2 with
// 256 threads making three dependent passes).
constexpr int kRowThreads = 1024, kRowValues = 8;

__device__ __forceinline__ float block_reduce(float v, float *red, bool is_max) {
  v = is_max ? col_max(row_max(v)) : col_sum(row_sum(v));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  v = red[threadIdx.x & 15];  // one value per wave
  v = is_max ? row_max(v) : row_sum(v);
  __syncthreads();
  return v;
}

__global__ __launch_bounds__(kRowThreads) void model_softmax_kernel(ModelAttnParams p) {
  static_assert(kRowThreads == 16 * 64, "block_reduce: 16 waves");
  __shared__ float red[16];
  const int64_t r = blockIdx.x;
  const int tid = threadIdx.x;
  const int end = min(p.tokens, p.start + (int)(r / p.q_heads) + 1);
  const float *lg = p.scores + r * p.tokens;
  float *pr = p.probs + r * p.tokens;
  constexpr int kSpan = kRowThreads * kRowValues;
  float x[kRowValues];
  float m = -3.4e38f, s = 0.0f;
  // The first kSpan tokens in registers.
#pragma unroll
  for (int k = 0; k < kRowValues; ++k) {
    const int t = tid + k * kRowThreads;
    x[k] = k * kRowThreads < end ? lg[t < end ? t : 0] : 0.0f;
  }
#pragma unroll
  for (int k = 0; k < kRowValues; ++k)
    if (tid + k * kRowThreads < end) m = fmaxf(m, x[k]);
  for (int t = tid + kSpan; t < end; t += kRowThreads) m = fmaxf(m, lg[t]);
  m = block_reduce(m, red, true);
#pragma unroll
  for (int k = 0; k < kRowValues; ++k) {
    if (k * kRowThreads >= end) break;  // uniform
    x[k] = tid + k * kRowThreads < end ? expf(x[k] - m) : 0.0f;
    s += x[k];
  }
  for (int t = tid + kSpan; t < end; t += kRowThreads) s += expf(lg[t] - m);
  s = block_reduce(s, red, false);
#pragma unroll
  for (int k = 0; k < kRowValues; ++k) {
    const int t = tid + k * kRowThreads;
    if (k * kRowThreads >= p.tokens) break;  // uniform
    if (t < p.tokens) pr[t] = (t < end ? x[k] : 0.0f) / s;
  }
  for (int t = tid + kSpan; t < p.tokens; t += kRowThreads) pr[t] = (t < end ? expf(lg[t] - m) : 0.0f) / s;
}

// attention.wgsl:32-39: output[r][dm] = sum_{t < end} p[r][t] v[kv][t][dm],
// kv = (r mod qHeads) / gqa: a [query items x tokens] x [tokens x d] product,
// the items of a KV head being its row-major rows x gqa. Two kernels, so that
// few items and many both spread over the chip and the sum over the tokens
// is short chains side by side: 9 heads x 4097 tokens 8.0 us, 288 rows x
// 2048 tokens 15.3 us (one workgroup per score row, its waves walking 1024
// tokens each: 100 and 52 us). Forming the probabilities in this kernel as
// well (no softmax launch) measured slower, 22-27 us: its few workgroups
// took every exponential twice over.

// Up to kFewItems items (a decode step's): a workgroup per KV head and four
// dimensions, a thread per token, on the vector ALUs (a matrix-core tile
// would be mostly padding). Grid: (d / 4, KV heads).
// Eight waves: the loads of nine tokens a thread in flight cover 4608 tokens
// in one round trip, and the reductions at the end (a wave's worth of
// instructions each) share a SIMD with one other wave (9 heads x 4097
// tokens: 8.0 us, 8.9 with 16 waves of five tokens); longer histories take
// more rounds (a whole SmolLM2 layer's dispatches, us, general kernels / these: 1
// row after 4096 tokens 290 / 62, 9000 420 / 70, 16,000 1112 / 91, 40,000 2970 / 143).
constexpr int kFewItems = 4, kFewThreads = 512;

template <bool ALIGNED>
__global__ __launch_bounds__(kFewThreads) void model_weighted_few_kernel(ModelAttnParams p) {
  constexpr int kWaves = kFewThreads / 64, U = 9, kBatch = U * kFewThreads;
  __shared__ float part[kWaves][kFewItems * 4];
  const int tid = threadIdx.x, kv = blockIdx.y, G = p.gqa, n_items = p.rows * G;
  auto score_row = [&](int item) { return (int64_t)(item / G) * p.q_heads + kv * G + item % G; };
  const int end_hi = min(p.tokens, p.start + (n_items - 1) / G + 1);
  const float *pr[kFewItems];
  int end[kFewItems];
#pragma unroll
  for (int k = 0; k < kFewItems; ++k) {
    const int64_t r = score_row(min(k, n_items - 1));
    const bool active = k < n_items && r < p.score_rows;
    end[k] = active ? min(p.tokens, p.start + k / G + 1) : 0;
    pr[k] = p.probs + (active ? r * p.tokens : 0);
  }
  const uint16_t *vh = p.v + (int64_t)kv * p.capacity * p.dim + 4 * blockIdx.x;
  const int vrow = p.dim * 2;
  float acc[kFewItems][4] = {};
  // Buffer ranges end at the causal ends: loads past them give zeros.
  for (int b0 = 0; b0 < end_hi; b0 += kBatch) {
    u32x2 v[U];
    float x[kFewItems][U];
    const __amdgpu_buffer_rsrc_t rv = rsrc(vh + (int64_t)b0 * p.dim, (uint32_t)((min(end_hi - b0, kBatch) - 1) * vrow + 8));
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int off = (tid + u * kFewThreads) * vrow;
      if (ALIGNED) {
        v[u] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rv, off, 0, 0));
      } else {
        uint32_t h[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) h[i] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rv, off + 2 * i, 0, 0);
        v[u] = u32x2{h[0] | h[1] << 16, h[2] | h[3] << 16};
      }
    }
#pragma unroll
    for (int k = 0; k < kFewItems; ++k) {
      if (k >= n_items) break;  // uniform
      const __amdgpu_buffer_rsrc_t rp = rsrc(pr[k] + b0, (uint32_t)max(0, min(end[k] - b0, kBatch)) * 4u);
#pragma unroll
      for (int u = 0; u < U; ++u)
        x[k][u] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rp, (tid + u * kFewThreads) * 4, 0, 0));
    }
#pragma unroll
    for (int k = 0; k < kFewItems; ++k) {
      if (k >= n_items) break;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        // (several rows: a V value past this row's end, perhaps not finite)
        if (p.rows > 1 && b0 + tid + u * kFewThreads >= end[k]) continue;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          acc[k][i] = __builtin_fmaf(x[k][u], h2f((uint16_t)(v[u][i >> 1] >> (16 * (i & 1)))), acc[k][i]);
      }
    }
  }
#pragma unroll
  for (int k = 0; k < kFewItems; ++k) {
    if (k >= n_items) break;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float o = col_sum(row_sum(acc[k][i]));
      if ((tid & 63) == 0) part[tid >> 6][4 * k + i] = o;
    }
  }
  __syncthreads();
  if (tid < 4 * n_items) {
    float o = 0.0f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) o += part[w][tid];
    const int64_t at = score_row(tid >> 2) * p.dim + 4 * blockIdx.x + (tid & 3);
    if (at < p.x_limit) p.out[at] = o;
  }
}

// More items: 16 items by 16 dimensions a workgroup, in FP32 on the matrix
// cores (16x16x4), its eight waves taking every eighth block of 16 tokens
// and meeting in LDS; the items' probabilities come through LDS (kChunk
// tokens at a time, within the LDS of one workgroup). Bound: the products and one memory round trip per four
// blocks of V. A whole SmolLM2 layer's dispatches, us, general kernels / these: 32 rows
// after 10 tokens 186 / 65, 2016 240 / 78, 4064 310 / 101, 8000 705 / 136; 200
// rows after 4000 768 / 180. Grid: (d / 16, tiles of 16 items, KV heads).
constexpr int kWeightedWaves = 8, kProbChunk = 2176, kProbRow = kProbChunk + 4;
constexpr int kProbBytes = 16 * kProbRow * 4;

__global__ __launch_bounds__(64 * kWeightedWaves) void model_weighted_kernel(ModelAttnParams p) {
  __shared__ float part[kWeightedWaves][256];
  extern __shared__ __align__(16) uint8_t smem[];
  float *prob = reinterpret_cast<float *>(smem);  // [item][kRow]
  constexpr int kChunk = kProbChunk, kRow = kProbRow;
  static_assert(kProbBytes + (int)sizeof(part) <= kLdsLimit, "LDS of one workgroup");
  static_assert(kChunk % 64 == 0, "whole runs of 64 tokens");
  const int tid = threadIdx.x, lane = tid & 63, gq = lane >> 4, col = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform: scalar addresses and loops
  const int slice = blockIdx.x, kv = blockIdx.z, G = p.gqa;
  const int i0 = blockIdx.y * 16, n_items = min(16, p.rows * G - i0);
  auto score_row = [&](int item) { return (int64_t)(item / G) * p.q_heads + kv * G + item % G; };
  auto end_of = [&](int item) { return min(p.tokens, p.start + item / G + 1); };
  const int end_lo = end_of(i0), end_hi = end_of(i0 + n_items - 1);
  constexpr int kStaged = 16 / kWeightedWaves;  // items a wave stages
  const uint16_t *vh = p.v + (int64_t)kv * p.capacity * p.dim;
  const float *prow = prob + col * kRow + 4 * gq;
  const int vrow = p.dim * 2, voff = 4 * gq * vrow + 32 * slice + 2 * col;
  f32x4 acc = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  constexpr int U = 4;
  for (int c0 = 0; c0 < end_hi; c0 += kChunk) {
    if (c0 > 0) __syncthreads();
    const int n_blocks = (min(kChunk, end_hi - c0) + 15) / 16;
    // This wave's items to LDS: zeros past the causal end, for rows the
    // dispatch does not cover and for those past the items.
#pragma unroll
    for (int h = 0; h < kStaged; ++h) {
      const int k = wave + h * kWeightedWaves;
      const int64_t r = score_row(i0 + min(k, n_items - 1));
      const int end = k < n_items && r < p.score_rows ? end_of(i0 + k) : 0;
      const __amdgpu_buffer_rsrc_t rx = rsrc(p.probs + (end ? r * p.tokens + c0 : 0), (uint32_t)max(0, min(end - c0, kChunk)) * 4u);
#pragma clang loop unroll(disable)
      for (int t = 0; t < 16 * n_blocks; t += 64)
        dma4(rx, reinterpret_cast<uint8_t *>(prob + k * kRow + t), (uint32_t)(t + lane) * 4u, 0);
    }
    // The V rows of block b + u kWeightedWaves: a range of the chunk's tokens
    // before the last causal end, zeros past it and for blocks past the last.
    auto load_v = [&](int b, uint16_t (&v)[U][4]) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int tb = 16 * (b + u * kWeightedWaves);
        const int rows = max(0, min(min(end_hi - c0, kChunk) - tb, 16));
        const __amdgpu_buffer_rsrc_t rv = rsrc(vh + (int64_t)(rows ? c0 + tb : 0) * p.dim, (uint32_t)(rows * vrow));
#pragma unroll
        for (int i = 0; i < 4; ++i) v[u][i] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rv, voff + i * vrow, 0, 0);
      }
    };
    uint16_t v[U][4], vn[U][4];
    load_v(wave, v);
    wait_vm<0>();  // the staged rows
    __syncthreads();
#pragma clang loop unroll(disable)
    for (int b = wave; b < n_blocks; b += U * kWeightedWaves) {
      load_v(b + U * kWeightedWaves, vn);
      f32x4 pr[U];
#pragma unroll
      for (int u = 0; u < U; ++u)
        pr[u] = *reinterpret_cast<const f32x4 *>(prow + 16 * min(b + u * kWeightedWaves, n_blocks - 1));
      bool odd = false;  // a V value that is not finite, in blocks past the first row's causal end
      if (c0 + 16 * (b + U * kWeightedWaves) > end_lo) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i) odd |= (v[u][i] & 0x7c00u) == 0x7c00u;
      }
      if (__builtin_amdgcn_ballot_w64(odd)) {
        // A value that is not finite, perhaps among the chunk's own tokens: a
        // row whose causal end lies before it must not meet it, not even
        // weighted zero.
#pragma clang loop unroll(disable)
        for (int u = 0; u < U * 16; ++u) {
          const int tb = 16 * (b + (u >> 4) * kWeightedWaves) + (u & 15);
          if (b + (u >> 4) * kWeightedWaves >= n_blocks || c0 + tb >= end_hi) continue;  // wave-uniform
          const float vv = h2f(vh[(int64_t)(c0 + tb) * p.dim + 16 * slice + col]);
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const int it = min(4 * gq + k, n_items - 1);
            const float pp = prob[it * kRow + tb];
            if (c0 + tb < end_of(i0 + it)) acc[k] = __builtin_fmaf(pp, vv, acc[k]);
          }
        }
      } else {
        // (a block past the last would multiply the last one's probabilities,
        // perhaps infinite ones of the caller's, by zeros)
#pragma unroll
        for (int u = 0; u < U; ++u) {
          if (b + u * kWeightedWaves >= n_blocks) break;  // wave-uniform
#pragma unroll
          for (int i = 0; i < 4; ++i) acc = mfma_f32(pr[u][i], h2f(v[u][i]), acc);
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) v[u][i] = vn[u][i];
    }
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) part[wave][(4 * gq + k) * 16 + col] = acc[k];
  __syncthreads();
  if (tid < 16 * n_items) {
    const int64_t at = score_row(i0 + tid / 16) * p.dim + 16 * slice + tid % 16;
    float o = 0.0f;
#pragma unroll
    for (int w = 0; w < kWeightedWaves; ++w) o += part[w][tid];
    if (at < p.x_limit) p.out[at] = o;
  }
}

}  // namespace

hipError_t launch_model_append(const ModelAppendParams &p, hipStream_t stream) {
  if (p.pairs <= 0) return hipSuccess;
  hipLaunchKernelGGL(model_append_kernel, dim3((unsigned)((p.pairs + 255) / 256)), dim3(256), 0, stream, p);
  return hipGetLastError();
}

namespace {
template <int D, int KF>
hipError_t launch_scores(const ModelScoresParams &p, int kv_count, int book_bytes, hipStream_t stream) {
  // The books may take the workgroup past the default 64 KB of LDS.
  static const hipError_t allowed = hipFuncSetAttribute((const void *)model_scores_kernel<D, KF>,
                                                        hipFuncAttributeMaxDynamicSharedMemorySize, 64 * 1024);
  if (allowed != hipSuccess) {
    (void)hipGetLastError();
    return allowed;
  }
  const dim3 grid((unsigned)((p.n_tok + kScoreTokens - 1) / kScoreTokens),
                  (unsigned)((p.rows * p.gqa + kScoreItems - 1) / kScoreItems), (unsigned)kv_count);
  hipLaunchKernelGGL((model_scores_kernel<D, KF>), grid, dim3(256), book_bytes, stream, p);
  return hipGetLastError();
}
}  // namespace

hipError_t launch_model_scores(const ModelScoresParams &p, int kv_count, int book_bytes, hipStream_t stream) {
  if (p.n_tok <= 0 || p.rows <= 0 || kv_count <= 0) return hipSuccess;
  if (p.k) return p.dim == 64 ? launch_scores<64, 0>(p, kv_count, 0, stream) : launch_scores<128, 0>(p, kv_count, 0, stream);
  return p.dim == 64 ? launch_scores<64, 1>(p, kv_count, book_bytes, stream)
                     : launch_scores<128, 1>(p, kv_count, book_bytes, stream);
}

hipError_t launch_model_softmax(const ModelAttnParams &p, hipStream_t stream) {
  if (p.score_rows <= 0) return hipSuccess;
  hipLaunchKernelGGL(model_softmax_kernel, dim3((unsigned)p.score_rows), dim3(kRowThreads), 0, stream, p);
  return hipGetLastError();
}

hipError_t launch_model_weighted(const ModelAttnParams &p, hipStream_t stream) {
  if (p.score_rows <= 0) return hipSuccess;
  const int64_t items = (int64_t)p.rows * p.gqa;
  const unsigned kvh = (unsigned)(p.q_heads / p.gqa);
  if (items <= kFewItems) {
    const dim3 grid((unsigned)(p.dim / 4), kvh);
    if (reinterpret_cast<uintptr_t>(p.v) % 8 == 0)
      hipLaunchKernelGGL(model_weighted_few_kernel<true>, grid, dim3(kFewThreads), 0, stream, p);
    else
      hipLaunchKernelGGL(model_weighted_few_kernel<false>, grid, dim3(kFewThreads), 0, stream, p);
    return hipGetLastError();
  }
  static const hipError_t allowed = hipFuncSetAttribute((const void *)model_weighted_kernel,
                                                        hipFuncAttributeMaxDynamicSharedMemorySize, kProbBytes);
  if (allowed != hipSuccess) {
    (void)hipGetLastError();
    return allowed;
  }
  const dim3 grid((unsigned)(p.dim / 16), (unsigned)((items + 15) / 16), kvh);
  hipLaunchKernelGGL(model_weighted_kernel, grid, dim3(64 * kWeightedWaves), kProbBytes, stream, p);
  return hipGetLastError();
}

}  // namespace bgtq
