// Bulk Block-GTQ K encode for gfx950, 16 rows per wave with the group
// rotations on the FP32 matrix cores: any layout whose groups are ascending
// contiguous runs of the head-perm order with even boundaries (every layout
// of paired widths). Bit-exact with the reference encoder
// (src/reference/production_math.py:4-24) under the contract of encode.hip:
//  * y_j = sum_i xn_i R[j][i] (production_math.py:16) is one FMA chain over i
//    in ascending order from +0. v_mfma_f32_16x16x4_f32 is that chain: its
//    four products enter the accumulator one FMA after another in ascending k
//    (2^20 random results, magnitudes 10^-40 to 10^40 and signed zeros
//    among them, all equal to fmaf chains bit for bit), so the products of
//    consecutive 4-wide steps continue it. Off-group entries of R are exact
//    zeros (validated when the tables are built), and steps whose 16 x 4
//    block is all zeros are skipped;
//  * the FP32 sums of production_math.py:12, :14 and :23 follow ATen's 8-lane
//    inner-sum tree: position 8 v + l enters lane l's accumulator v mod 4,
//    then ((a0 + a1) + a2) + a3, then the eight lanes in order. The leaves
//    outside a group are +0 and the accumulators never negative, so leaving
//    them out changes nothing;
//  * division and square root are IEEE (-ffp-contract=off, correctly rounded);
//    the divisions by a group's norm use its correctly rounded reciprocal and
//    one FMA correction, which gives the same quotients
//    (tests/host_division_check.c).
//
// Lane (gq, col) = (lane / 16, lane % 16) holds a quarter of row col, the
// positions 4 s + gq: inputs as the product's B operand (step s = 4 t + r),
// outputs as its result (row 4 gq + r of tile t is position 16 t + 4 r + gq,
// an order the A operand is free to choose). A lane so holds whole columns
// l = gq and 4 + gq of the sum tree. The masked sums of four groups at once
// are 4x4x1 matrix products (one exact FMA per leaf and group); a 4 x 4
// transpose by row swaps then gives lane gq the eight partials of group gq,
// so each group's square roots and divisions are taken once per row; a
// 16x16x4 product with 0/1 masks hands every position its group's divisor.
//
// Bound: the matrix cores (about 60 products of 32 cycles per 16 rows at d=64
// and four groups), the LDS reads of their operands and of the code table,
// and the vector instructions take about equal time. 368,640 rows of the 90
// SmolLM2 calibration heads: 77 us, 331 with a thread per row (encode.hip);
// 262,144 rows of layout B 45 us, 48 with its compile-time structure
// (encode_bulk.hip, ahead where its rounds of 196,608 rows are well filled: 29
// against 37.5 us for 196,608, 51 against 57 for 368,640); d=128 layouts 103-117 us for 184,320 rows, 137 and 624 before.
#include <hip/hip_fp16.h>

#include "bgtq_internal.h"
#include "encode_row.h"
#include "gfx950_common.h"

namespace bgtq {
namespace {

using namespace gfx;
using row_enc::f16_bits_to_f32;
using row_enc::f32_to_f16_bits;
using row_enc::wave_sync;

// Tables and job read through the constant address space: nothing writes them
// while the kernel runs, so their wave-uniform fields are scalar loads.
#define BGTQ_CONST __attribute__((address_space(4)))
template <typename X>
__device__ __forceinline__ const BGTQ_CONST X *to_const(const void *p) {
  return (const BGTQ_CONST X *)reinterpret_cast<uintptr_t>(p);
}

constexpr int kTileRows = 16;
constexpr int tile_waves(int D) { return D == 64 ? 4 : 8; }

// LDS of a workgroup: the rotation as A operands, the combined code table
// ({centroid squared, code} per codebook and bin), per-position constants,
// the groups' masks and leaf counts, then per wave one block's rows (first
// the inputs, then the packed rows' image). Sized for the launch's largest
// codebook count, group count and row bytes.
struct TileLds {
  int tab, pos, cnt, mask, sel, src, wave, dump, stride, total;
};
template <int D>
struct Tile {
  static constexpr int KS = D / 4, NT = D / 16, NV = D / 8;
  static constexpr int MROW = KS + 4;          // floats per mask row
  static constexpr int XROW = 2 * D + 8;       // bytes per staged input row
  static constexpr int PROW = 2 * KS + 4;      // floats per lane group of off/inv
};
template <int D>
__host__ __device__ inline TileLds tile_lds(int n_codebooks, int groups, int row_bytes) {
  using S = Tile<D>;
  TileLds L;
  const int gb = (groups + 3) / 4;
  int o = D * D * 4;  // A operands at 0
  L.tab = o; o += n_codebooks * 256 * 8;
  L.pos = o; o += 4 * S::PROW * 4;                  // [gq][s]: off, inv
  L.src = o; o += 4 * S::MROW * 4;                  // [gq][s]: source byte of position 4 s + gq | codebook << 16
  L.cnt = o; o += groups * 32 * (D == 64 ? 4 : 8);  // [group][l][k]
  L.mask = o; o += gb * 16 * S::MROW * 4;           // [block of 4 groups][gq][group][s]
  L.sel = o; o += gb * 64 * (S::NT + (S::NT == 4 ? 0 : 4)) * 4;  // [block][lane][t]
  L.wave = o;
  const int img = kTileRows * row_bytes + 4, x = kTileRows * S::XROW;
  L.dump = (img > x ? img : x) / 16 * 16 + 16;  // where nibble lanes put a second byte
  L.stride = L.dump + 16;
  L.total = o + tile_waves(D) * L.stride;
  return L;
}

// Waves per SIMD that the register budget leaves room for.
constexpr int tile_waves_per_simd(int D, bool src_f32) { return D != 64 ? 2 : src_f32 ? 3 : 4; }

// One job: its packed and norms already point at its first destination row.
//
// The products with 0/1 masks below spread an infinity or a NaN over every
// group of its row (0 inf = NaN). A wave that met one encodes those of its
// blocks again after its loop, with selects, as the other encoders do: a
// group's norm takes its own inputs, and its y are NaN (bin 0) when their FMA
// chain meets a non-finite input. The chain runs over the 8-wide blocks that
// touch the group (encode.hip; whole groups in encode_bulk.hip), or with
// WHOLE_ROWS over the row (the wave encoder, for smaller calls).
template <int D, bool SRC_F32, bool WHOLE_ROWS>
__device__ __forceinline__ void encode_tile_body(const EncodeTileJob &job, const int64_t rows, int max_codebooks,
                                                 int max_groups, int max_row_bytes) {
  using S = Tile<D>;
  constexpr int KS = S::KS, NT = S::NT, NV = S::NV, W = tile_waves(D), TH = 64 * W;
  constexpr int kSelRow = NT + (NT == 4 ? 0 : 4);
  extern __shared__ __align__(16) uint8_t smem[];
  const TileLds L = tile_lds<D>(max_codebooks, max_groups, max_row_bytes);
  const int64_t n_blocks = (rows + kTileRows - 1) / kTileRows;
  if ((int64_t)blockIdx.x * W >= n_blocks) return;  // uniform for the workgroup
  const BGTQ_CONST DevTables *T = to_const<DevTables>(job.t);
  const int tid = threadIdx.x, lane = tid & 63, gq = lane >> 4, col = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ng = T->groups, ngb = (ng + 3) / 4, mc = T->max_centroids, ns = T->nibble_dims, RB = T->row_bytes,
            NS = T->norm_stride;
  float *const a_op = reinterpret_cast<float *>(smem);
  float *const cnt = reinterpret_cast<float *>(smem + L.cnt);
  uint8_t *const wv = smem + L.wave + wave * L.stride;
  // The image of a block's packed rows starts at the destination's byte in
  // its word (the same for every block: 16 rows are whole words).
  const uint32_t mis = (uint32_t)reinterpret_cast<uintptr_t>(job.packed) & 3u;

  // A quarter of row col of block b per lane, in 16-byte pieces where the
  // source allows, through a buffer range that ends with the job's last row
  // (rows past it read as zeros and are not stored). FP32 sources are rounded
  // to FP16 first (src/model/codec.wgsl:14).
  constexpr int kElem = SRC_F32 ? 4 : 2, NP = KS * kElem / 16;  // 16-byte pieces per lane
  const bool vec = reinterpret_cast<uintptr_t>(job.src) % 16 == 0 && (job.src_stride * kElem) % 16 == 0;  // uniform
  u32x4 raw[NP];
  auto load_rows = [&](int64_t b, int gq, int col) {
    const int nr = (int)min((int64_t)kTileRows, rows - b * kTileRows);
    const uint8_t *base = static_cast<const uint8_t *>(job.src) + b * kTileRows * (int64_t)job.src_stride * kElem;
    const __amdgpu_buffer_rsrc_t r =
        rsrc(nr > 0 ? base : job.src, nr > 0 ? (uint32_t)((nr - 1) * job.src_stride + D) * kElem : 0u);
    const uint32_t at = (uint32_t)(col * job.src_stride + KS * gq) * kElem;
    if (vec) {
#pragma unroll
      for (int k = 0; k < NP; ++k)
        raw[k] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)(at + 16 * k), 0, 0));
    } else if (SRC_F32) {
#pragma unroll
      for (int k = 0; k < 4 * NP; ++k) raw[k / 4][k % 4] = __builtin_amdgcn_raw_buffer_load_b32(r, (int)(at + 4 * k), 0, 0);
    } else {
#pragma unroll
      for (int k = 0; k < 4 * NP; ++k) {
        const uint32_t lo = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(r, (int)(at + 4 * k), 0, 0);
        const uint32_t hi = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(r, (int)(at + 4 * k + 2), 0, 0);
        raw[k / 4][k % 4] = lo | hi << 16;
      }
    }
  };
  // The loaded rows to LDS as FP16, in natural order; the lanes whose part
  // holds an infinity or a NaN (FP16 squares sum to at most 3e11).
  auto stage_rows = [&](int gq, int col) {
    float squares = 0.0f;
#pragma unroll
    for (int k = 0; k < KS / 4; ++k) {
      uint32_t v[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int c = 4 * k + 2 * h;
        if (SRC_F32)
          v[h] = (uint32_t)f32_to_f16_bits(__uint_as_float(raw[c / 4][c % 4])) |
                 (uint32_t)f32_to_f16_bits(__uint_as_float(raw[c / 4][c % 4 + 1])) << 16;
        else
          v[h] = raw[k / 2][2 * (k % 2) + h];
        typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
        const half2_t x = __builtin_bit_cast(half2_t, v[h]);
        squares = __builtin_amdgcn_fdot2(x, x, squares, false);
      }
      *reinterpret_cast<u32x2 *>(wv + col * S::XROW + 2 * KS * gq + 8 * k) = u32x2{v[0], v[1]};
    }
    return __builtin_amdgcn_ballot_w64(!(squares < INFINITY));
  };
  uint64_t odd_seen = 0;
  const int64_t b_first = (int64_t)blockIdx.x * W + wave;
  load_rows(b_first, gq, col);

  // ---- the workgroup's tables ----
  const uint8_t *Tg = reinterpret_cast<const uint8_t *>(job.t);
  {
    const uint8_t *perm = Tg + offsetof(DevTables, perm), *grp = Tg + offsetof(DevTables, group_of),
                  *pcb = Tg + offsetof(DevTables, pos_cb), *pbk = Tg + offsetof(DevTables, pos_book);
    const float *loff = reinterpret_cast<const float *>(Tg + offsetof(DevTables, lut_off)),
                *linv = reinterpret_cast<const float *>(Tg + offsetof(DevTables, lut_inv));
    for (int p = tid; p < D; p += TH) {  // position p = 4 s + gq
      const int q = p & 3, i = p >> 2;
      reinterpret_cast<uint32_t *>(smem + L.src)[q * S::MROW + i] = (uint32_t)perm[p] * 2u | (uint32_t)pcb[p] << 16;
      float *f = reinterpret_cast<float *>(smem + L.pos) + q * S::PROW + 2 * i;
      f[0] = loff[p];
      f[1] = linv[p];
    }
    // A codebook's centroids are those of its first position (64 positions'
    // codebooks per ballot; a wave's 64 bins lie in one codebook).
    const uint8_t *lut = Tg + T->off_lut;
    const float *books = reinterpret_cast<const float *>(Tg + T->off_books);
    const uint32_t cb0 = pcb[lane], cb1 = D > 64 ? pcb[64 + lane] : 0u;
    for (int e = tid; e < T->n_codebooks * 256; e += TH) {
      const uint32_t code = lut[e];
      const uint64_t f0 = __builtin_amdgcn_ballot_w64(cb0 == (uint32_t)(e >> 8)),
                     f1 = D > 64 ? __builtin_amdgcn_ballot_w64(cb1 == (uint32_t)(e >> 8)) : 0u;
      const int p = f0 ? __builtin_ctzll(f0) : f1 ? 64 + __builtin_ctzll(f1) : 0;
      const float c = books[(int)pbk[p] * mc + (int)code];
      reinterpret_cast<u32x2 *>(smem + L.tab)[e] = u32x2{__float_as_uint(c * c), code};
    }
    const float *R = reinterpret_cast<const float *>(Tg + T->off_rot);
    for (int e = tid; e < D * D / 4; e += TH) {
      // Row j = 16 t + 4 r + q (operand row m = 4 q + r of tile t), columns
      // i .. i + 3 (k = 0..3 of step i / 4).
      const int j = e / (D / 4), i = 4 * (e % (D / 4)), t = j / 16, m = 4 * (j & 3) + ((j >> 2) & 3);
      const f32x4 v = *reinterpret_cast<const f32x4 *>(R + j * D + i);
#pragma unroll
      for (int k = 0; k < 4; ++k) a_op[((t * NT + i / 16) * 64 + 16 * k + m) * 4 + (i % 16) / 4] = v[k];
    }
    // Group masks (1 or 0): of the tree's leaves, as lane 4 b + i of the 4x4
    // blocks (16 lanes per gq) holds group i's; of the positions, as the A
    // operand (row m = 4 q + r of tile t: position 16 t + 4 r + q; column k:
    // group k) of the product that selects each position's group.
    for (int e = tid; e < ngb * 16 * KS; e += TH) {
      const int r = e / KS, i = e % KS, g = r / 16 * 4 + (r & 3), p = 4 * i + ((r >> 2) & 3);
      reinterpret_cast<float *>(smem + L.mask)[r * S::MROW + i] = grp[p] == g ? 1.0f : 0.0f;
    }
    for (int e = tid; e < ngb * 64 * NT; e += TH) {
      const int t = e % NT, l = e / NT, m = l & 15, g = l / 64 * 4 + ((l >> 4) & 3), p = 16 * t + 4 * (m & 3) + (m >> 2);
      reinterpret_cast<float *>(smem + L.sel)[l * kSelRow + t] = grp[p] == g ? 1.0f : 0.0f;
    }
    for (int e = tid; e < ng * 32; e += TH) {  // leaves of group g at lane l, accumulator k
      const int g = e / 32, l = (e / 4) % 8, k = e % 4;
      int c = 0;
#pragma unroll
      for (int v = 0; v < NV; v += 4) c += grp[8 * (v + k) + l] == g;
      if (D == 64) {
        cnt[e] = (float)c;
      } else {
        cnt[2 * e] = (float)min(c, 3);
        cnt[2 * e + 1] = c > 3 ? 1.0f : 0.0f;
      }
    }
    __syncthreads();
  }
  // The 4-wide steps each tile of 16 positions needs, in groups of four.
  int qlo[NT], qhi[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    qlo[t] = T->gstart[T->group_of[16 * t]] / 16;
    qhi[t] = (T->gend[T->group_of[16 * t + 15]] - 1) / 16;
  }
  // The transpose over the four rows of lanes: v[i] of lane group q becomes
  // v[q] of lane group i.
  auto transpose4 = [&](f32x4 &v) {
    auto sw32 = [&](int i, int j) {
      auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[i]), __float_as_uint(v[j]), false, false);
      v[i] = __uint_as_float(r[0]);
      v[j] = __uint_as_float(r[1]);
    };
    auto sw16 = [&](int i, int j) {
      auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[i]), __float_as_uint(v[j]), false, false);
      v[i] = __uint_as_float(r[0]);
      v[j] = __uint_as_float(r[1]);
    };
    sw32(0, 2);
    sw32(1, 3);
    sw16(0, 1);
    sw16(2, 3);
  };
  for (int64_t b = b_first; b < n_blocks; b += (int64_t)gridDim.x * W) {
    // The lane index through an opaque copy: offsets derived from it are
    // recomputed where they are used instead of being held in registers
    // across the loop (which spilled: 45 registers at four waves per SIMD).
    int lane = tid & 63;
    asm volatile("" : "+v"(lane));
    const int gq = lane >> 4, col = lane & 15;
    // Where this lane's pairs of codes go in the rows' image
    // (mixed_layout.py:21-27). After the row swap below it holds, for each even
    // step s, the codes of positions 4 (s + (gq & 1)) + 2 (gq >> 1) + {0, 1}: a
    // nibble pair shares a byte (its second store goes nowhere), byte codes
    // take one each.
    auto pair_pos = [&](int s) { return 4 * (s + (gq & 1)) + 2 * (gq >> 1); };
    uint8_t *const img0 = wv + mis;
    const int row_at = col * RB;
    // ATen's 8-lane sum of this row's leaves (leaf(s): position 4 s + gq) over
    // group 4 h + gq: per column the four interleaved accumulators of each
    // group of block h, then the eight columns in order.
    const int mrow = 4 * gq + (lane & 3);  // this lane's row of the mask table
    auto tree_sum = [&](int h, auto leaf) {
      const f32x4 *mp = reinterpret_cast<const f32x4 *>(smem + L.mask + (16 * h + mrow) * S::MROW * 4);
      f32x4 m[KS / 4], p[2];
  #pragma unroll
      for (int q = 0; q < KS / 4; ++q) m[q] = mp[q];
  #pragma unroll
      for (int k = 0; k < 4; ++k)
  #pragma unroll
        for (int e = 0; e < 2; ++e) {
          f32x4 a = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  #pragma unroll
          for (int v = k; v < NV; v += 4) {
            const int i = 2 * v + e;
            a = __builtin_amdgcn_mfma_f32_4x4x1f32(m[i / 4][i % 4], leaf(i), a, 0, 0, 0);
          }
          p[e] = k == 0 ? a : p[e] + a;
        }
      transpose4(p[0]);
      transpose4(p[1]);
      return ((((((p[0][0] + p[0][1]) + p[0][2]) + p[0][3]) + p[1][0]) + p[1][1]) + p[1][2]) + p[1][3];
    };

    // The rows to LDS in natural order, the next block's loads, then this
    // lane's positions.
    odd_seen |= stage_rows(gq, col);
    load_rows(b + (int64_t)gridDim.x * W, gq, col);  // in flight meanwhile
    wave_sync();
    const u32x4 *so = reinterpret_cast<const u32x4 *>(smem + L.src + gq * S::MROW * 4);
    float x[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s)
      x[s] = f16_bits_to_f32(*reinterpret_cast<const uint16_t *>(wv + col * S::XROW + (so[s / 4][s % 4] & 0xffffu)));
    // production_math.py:12-15 for the row's groups gq and gq + 4: n_g,
    // raw_g = sum(n_g over the group)/|g|; then every position's divisor and
    // its reciprocal.
    float raw_g[2] = {0.0f, 0.0f};
    f32x4 den[NT], rcp[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) den[t] = rcp[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    for (int h = 0; h < ngb; ++h) {
      const int g = min(gq + 4 * h, ng - 1);
      const float n = __builtin_sqrtf(tree_sum(h, [&](int s) { return x[s] * x[s]; }) + 1e-30f);
      float rg = n;
      if (ng > 1) {
        // Accumulator k of lane l holds c leaves: n, 2n, 3n in one rounding,
        // and (3n) + n for the fourth (d=128).
        const f32x4 *cp = reinterpret_cast<const f32x4 *>(cnt + g * 32 * (D == 64 ? 1 : 2));
        float t = 0.0f;
#pragma unroll
        for (int l = 0; l < 8; ++l) {
          float pl;
          if (D == 64) {
            const f32x4 c = cp[l];
            pl = c[0] * n;
#pragma unroll
            for (int k = 1; k < 4; ++k) pl = __builtin_fmaf(c[k], n, pl);
          } else {
            const f32x4 c = cp[2 * l], d = cp[2 * l + 1];
            pl = __builtin_fmaf(c[1], n, c[0] * n);
            pl += __builtin_fmaf(c[3], n, c[2] * n);
            pl += __builtin_fmaf(d[1], n, d[0] * n);
            pl += __builtin_fmaf(d[3], n, d[2] * n);
          }
          t = l == 0 ? pl : t + pl;
        }
        rg = t / (float)T->gsize[g];
      }
      raw_g[0] = h == 0 ? rg : raw_g[0];
      raw_g[1] = h == 0 ? raw_g[1] : rg;
      const float dg = n > 1e-10f ? n : 1.0f, rd = 1.0f / dg;
      const float *sp = reinterpret_cast<const float *>(smem + L.sel) + (64 * h + lane) * kSelRow;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        den[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(sp[t], dg, den[t], 0, 0, 0);
        rcp[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(sp[t], rd, rcp[t], 0, 0, 0);
      }
    }
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const float r = rcp[s / 4][s % 4], q0 = x[s] * r;
      x[s] = __builtin_fmaf(__builtin_fmaf(-q0, den[s / 4][s % 4], x[s]), r, q0);
    }
    // The image's padding bytes (mixed_layout.py:21-27) over the input rows.
    wave_sync();
    if (RB > (ns >> 1) + D - ns)
      for (int o = lane; 4 * o < (int)mis + kTileRows * RB; o += 64) reinterpret_cast<uint32_t *>(wv)[o] = 0u;
    // production_math.py:16-18: y, bin, code and centroid squared.
    float c2[KS];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      f32x4 y = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int q = 0; q < NT; ++q) {
        if (q < qlo[t] || q > qhi[t]) continue;  // uniform
        const f32x4 a = *reinterpret_cast<const f32x4 *>(a_op + ((t * NT + q) * 64 + lane) * 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) y = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], x[4 * q + i], y, 0, 0, 0);
      }
      const f32x4 *pf = reinterpret_cast<const f32x4 *>(smem + L.pos + (gq * S::PROW + 8 * t) * 4);
      const u32x4 cw = so[t];
      const f32x4 f[2] = {pf[0], pf[1]};  // off, inv of steps 4 t .. 4 t + 3
      uint32_t code[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float u = __builtin_amdgcn_fmed3f((y[r] - f[r / 2][2 * (r % 2)]) * f[r / 2][2 * (r % 2) + 1], 0.0f, 255.0f);
        const u32x2 entry = *reinterpret_cast<const u32x2 *>(smem + L.tab + ((cw[r] >> 16) * 2048u + 8u * (uint32_t)(int)u));
        c2[4 * t + r] = __uint_as_float(entry[0]);
        code[r] = entry[1];
      }
#pragma unroll
      for (int r = 0; r < 4; r += 2) {
        // Rows of lanes 0, 1 (2, 3) hold the first and second code of a
        // nibble pair: the even row takes step s's pair, the odd one s + 1's.
        auto w = __builtin_amdgcn_permlane16_swap(code[r], code[r + 1], false, false);
        const int p = pair_pos(4 * t + r);
        const bool nib = p < ns;
        const int at = row_at + (nib ? p >> 1 : (ns >> 1) + p - ns);
        img0[at] = (uint8_t)(w[0] | w[1] << (nib ? 4 : 8));
        *(nib ? wv + L.dump : img0 + at + 1) = (uint8_t)w[1];
      }
    }
    // production_math.py:20-23: corrected_g = raw_g / max(sqrt(sum c^2), 1e-10).
    const int64_t row0 = b * kTileRows;
    const int nr = (int)min((int64_t)kTileRows, rows - row0);
    BGTQ_GLOBAL uint16_t *nrow = to_global(job.norms) + (row0 + col) * NS;
    for (int h = 0; h < ngb; ++h) {
      const int g = gq + 4 * h;
      const float c = fmaxf(__builtin_sqrtf(tree_sum(h, [&](int s) { return c2[s]; })), 1e-10f);
      const uint16_t sc = f32_to_f16_bits((h == 0 ? raw_g[0] : raw_g[1]) / c);
      if (g < ng && col < nr) nrow[g] = sc;
    }
    for (int g = ng + gq; g < NS; g += 4)
      if (col < nr) nrow[g] = 0;
    wave_sync();
    // The image to the destination: whole words, then the bytes of the first
    // and last word when they are not whole.
    uint8_t *dst = job.packed + row0 * RB - mis;
    const int e1 = (int)mis + nr * RB, w0 = mis ? 1 : 0, w1 = e1 / 4;
    for (int w = w0 + lane; w < w1; w += 64)
      *reinterpret_cast<BGTQ_GLOBAL uint32_t *>(to_global(dst) + 4 * w) = reinterpret_cast<const uint32_t *>(wv)[w];
    if (mis || e1 % 4) {  // uniform; lanes 0..3: the first word, 4..7: the last
      const int o = lane < 4 ? lane : 4 * w1 + lane - 4;
      if (lane < 4 ? mis && o >= (int)mis && o < e1 : lane < 8 && o < e1 && (w1 > 0 || !mis)) to_global(dst)[o] = wv[o];
    }
    wave_sync();  // the rows' LDS is rewritten by the next block
  }
  if (odd_seen == 0) return;

  // The blocks that hold infinities or NaNs once more, from their staged
  // rows: lane (gq, col) takes positions 4 s + gq of row col as above, so
  // columns gq and 4 + gq of the sum tree. Rolled loops: it is rare.
  wait_vm<0>();  // the stores below come after the loop's
  int odd_lane = lane_id();
  asm volatile("" : "+v"(odd_lane));  // (not held across the loop above)
  for (int64_t b = b_first; b < n_blocks; b += (int64_t)gridDim.x * W) {
    const int gq = odd_lane >> 4, col = odd_lane & 15;
    load_rows(b, gq, col);
    const uint64_t odd = stage_rows(gq, col);
    wave_sync();
    auto input = [&](int p) {
      return f16_bits_to_f32(*reinterpret_cast<const uint16_t *>(wv + col * S::XROW + 2 * (int)T->perm[p]));
    };
    // The tree's sum of leaf(p) over the positions p of [g0, g1).
    auto tree = [&](int g0, int g1, auto leaf) {
      float part[2];
#pragma clang loop unroll(disable)
      for (int h = 0; h < 2; ++h) {
        float t = 0.0f;
#pragma clang loop unroll(disable)
        for (int k = 0; k < 4; ++k) {
          float a = 0.0f;
#pragma clang loop unroll(disable)
          for (int v = k; v < NV; v += 4) {
            const int p = 8 * v + 4 * h + gq;
            const bool in = p >= g0 && p < g1;
            if (__builtin_amdgcn_ballot_w64(in) == 0) continue;
            const float x = leaf(p, in);
            a += in ? x : 0.0f;
          }
          t = k == 0 ? a : t + a;
        }
        part[0] = h == 0 ? t : part[0];
        part[1] = t;
      }
      float total = 0.0f;
      for (int l = 0; l < 8; ++l) {
        const float x = __shfl(l < 4 ? part[0] : part[1], 16 * (l & 3) + col, 64);
        total = l == 0 ? x : total + x;
      }
      return total;
    };
    const int64_t row = b * kTileRows + col;
    const bool stored = odd != 0 && row < rows;
    const float *R = reinterpret_cast<const float *>(Tg + T->off_rot);
    BGTQ_GLOBAL uint8_t *prow = to_global(job.packed) + row * RB;
    BGTQ_GLOBAL uint16_t *nrow = to_global(job.norms) + row * NS;
#pragma clang loop unroll(disable)
    for (int g = 0; g < (odd ? ng : 0); ++g) {
      const int g0 = T->gstart[g], g1 = T->gend[g];
      const int c0 = WHOLE_ROWS ? 0 : g0 & ~7, c1 = WHOLE_ROWS ? D : (g1 + 7) & ~7;
      const float n = __builtin_sqrtf(tree(g0, g1, [&](int p, bool) { return input(p) * input(p); }) + 1e-30f);
      const float rg = ng > 1 ? tree(g0, g1, [&](int, bool) { return n; }) / (float)T->gsize[g] : n;
      const float dg = n > 1e-10f ? n : 1.0f;
      const float s = tree(g0, g1, [&](int p, bool in) {
        float y = 0.0f;
#pragma clang loop unroll(disable)
        for (int i = c0; i < c1; ++i) {
          // An input of another group meets a zero of R: only one that is not finite counts.
          const float x = input(i);
          const float xn = i >= g0 && i < g1 ? x / dg : __builtin_fabsf(x) < INFINITY ? 0.0f : __builtin_nanf("");
          y = __builtin_fmaf(xn, R[p * D + i], y);
        }
        const float *f = reinterpret_cast<const float *>(smem + L.pos) + gq * S::PROW + 2 * (p >> 2);
        const uint32_t cb = reinterpret_cast<const uint32_t *>(smem + L.src)[gq * S::MROW + (p >> 2)] >> 16;
        const float u = fminf(fmaxf((y - f[0]) * f[1], 0.0f), 255.0f);
        const u32x2 e = *reinterpret_cast<const u32x2 *>(smem + L.tab + (cb * 2048u + 8u * (uint32_t)(int)u));
        // A nibble pair's lanes (gq even, odd) lie in one group; the even one stores the byte.
        const uint32_t other = (uint32_t)__shfl_xor((int)e[1], 16, 64);
        if (in && stored) {
          if (p >= ns) prow[(ns >> 1) + p - ns] = (uint8_t)e[1];
          else if (!(p & 1)) prow[p >> 1] = (uint8_t)(e[1] | other << 4);
        }
        return __uint_as_float(e[0]);
      });
      const uint16_t sc = f32_to_f16_bits(rg / fmaxf(__builtin_sqrtf(s), 1e-10f));
      if (gq == 0 && stored) nrow[g] = sc;
    }
    wave_sync();
  }
}

// Jobs from the context's device table, one per grid y.
template <int D, bool SRC_F32>
__global__ __launch_bounds__(64 * tile_waves(D), tile_waves_per_simd(D, SRC_F32)) void encode_tile_kernel(
    const EncodeJobDev *__restrict__ jobs, int max_codebooks, int max_groups, int max_row_bytes) {
  struct JobWords {
    u32x4 w[4];
  };
  const BGTQ_CONST u32x4 *jw = to_const<u32x4>(jobs + blockIdx.y);
  const EncodeJobDev j = __builtin_bit_cast(EncodeJobDev, (JobWords{{jw[0], jw[1], jw[2], jw[3]}}));
  const BGTQ_CONST DevTables *T = to_const<DevTables>(j.t);
  const EncodeTileJob job{j.t, j.src, j.packed + j.dst_row0 * T->row_bytes, j.norms + j.dst_row0 * T->norm_stride,
                          j.src_stride, 0};
  encode_tile_body<D, SRC_F32, false>(job, j.rows, max_codebooks, max_groups, max_row_bytes);
}

// Jobs from the kernel's arguments: small calls share no device memory with
// other calls on the context, and take no upload launch.
template <int D, bool SRC_F32>
__global__ __launch_bounds__(64 * tile_waves(D), tile_waves_per_simd(D, SRC_F32)) void encode_tile_args_kernel(
    EncodeTileLaunch launch, int max_codebooks, int max_groups, int max_row_bytes) {
  const EncodeTileJob job = launch.jobs[blockIdx.y];
  encode_tile_body<D, SRC_F32, true>(job, job.rows, max_codebooks, max_groups, max_row_bytes);
}

template <typename K, typename J>
hipError_t launch_k(K kernel, const hipError_t allowed, const dim3 grid, int threads, int lds, hipStream_t stream,
                    const J &jobs, const EncodeTileSizes &z) {
  if (allowed != hipSuccess) {
    (void)hipGetLastError();
    return allowed;
  }
  hipLaunchKernelGGL(kernel, grid, dim3((unsigned)threads), lds, stream, jobs, z.codebooks, z.groups, z.row_bytes);
  return hipGetLastError();
}

template <int D, bool SRC_F32>
hipError_t launch_d(const EncodeJobDev *table, const EncodeTileLaunch *args, const dim3 grid, const EncodeTileSizes &z,
                    hipStream_t stream) {
  const int lds = tile_lds<D>(z.codebooks, z.groups, z.row_bytes).total, threads = 64 * tile_waves(D);
  if (table) {
    static const hipError_t ok = hipFuncSetAttribute((const void *)encode_tile_kernel<D, SRC_F32>,
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, kLdsLimit);
    return launch_k(encode_tile_kernel<D, SRC_F32>, ok, grid, threads, lds, stream, table, z);
  }
  static const hipError_t ok = hipFuncSetAttribute((const void *)encode_tile_args_kernel<D, SRC_F32>,
                                                   hipFuncAttributeMaxDynamicSharedMemorySize, kLdsLimit);
  return launch_k(encode_tile_args_kernel<D, SRC_F32>, ok, grid, threads, lds, stream, *args, z);
}

hipError_t launch_any(const EncodeJobDev *table, const EncodeTileLaunch *args, int n_jobs, int dim, int src_f32,
                      int64_t max_rows, int cus, const EncodeTileSizes &z, hipStream_t stream) {
  const int64_t wg_rows = encode_tile_wg_rows(dim), most = (max_rows + wg_rows - 1) / wg_rows;
  const int64_t resident = encode_tile_resident(dim, src_f32, cus, z);
  const dim3 grid((unsigned)std::max<int64_t>(1, std::min<int64_t>(most, resident / n_jobs)), (unsigned)n_jobs);
  if (dim == 64)
    return src_f32 ? launch_d<64, true>(table, args, grid, z, stream) : launch_d<64, false>(table, args, grid, z, stream);
  return src_f32 ? launch_d<128, true>(table, args, grid, z, stream) : launch_d<128, false>(table, args, grid, z, stream);
}

}  // namespace

bool encode_tile_layout(const DevTables *T) {
  const int d = T->dim;
  if ((d != 64 && d != 128) || T->nibble_dims % 2) return false;
  for (int g = 0; g < T->groups; ++g)
    if (T->gstart[g] % 2 || T->gend[g] % 2 || T->gstart[g] != (g ? T->gend[g - 1] : 0)) return false;
  int book[256];
  for (int &x : book) x = -1;
  for (int j = 0; j < d; ++j) {  // one centroid book per codebook
    int &x = book[T->pos_cb[j]];
    if (x >= 0 && x != T->pos_book[j]) return false;
    x = T->pos_book[j];
  }
  return T->row_bytes <= 2 * d && encode_tile_lds_bytes(d, T->n_codebooks, T->groups, T->row_bytes) <= kLdsLimit;
}

int encode_tile_lds_bytes(int dim, int n_codebooks, int groups, int row_bytes) {
  return dim == 64 ? tile_lds<64>(n_codebooks, groups, row_bytes).total
                   : tile_lds<128>(n_codebooks, groups, row_bytes).total;
}

int encode_tile_wg_rows(int dim) { return kTileRows * tile_waves(dim); }

// One round of workgroups (as many waves per SIMD as their registers allow, as far as the LDS holds
// them) shared by the jobs, rounded down: a few more than fit take a second
// round as long as the first. A wave walks its job's blocks with that stride.
int64_t encode_tile_resident(int dim, int src_f32, int cus, const EncodeTileSizes &z) {
  const int lds = encode_tile_lds_bytes(dim, z.codebooks, z.groups, z.row_bytes);
  return (int64_t)cus * std::max(1, std::min(4 * tile_waves_per_simd(dim, src_f32) / tile_waves(dim), kLdsLimit / lds));
}

hipError_t launch_encode_tile(const EncodeJobDev *jobs, int n_jobs, int dim, int src_f32, int64_t max_rows, int cus,
                              const EncodeTileSizes &z, hipStream_t stream) {
  return launch_any(jobs, nullptr, n_jobs, dim, src_f32, max_rows, cus, z, stream);
}

hipError_t launch_encode_tile_args(const EncodeTileLaunch &launch, int dim, int src_f32, int64_t max_rows, int cus,
                                   const EncodeTileSizes &z, hipStream_t stream) {
  return launch_any(nullptr, &launch, launch.n_jobs, dim, src_f32, max_rows, cus, z, stream);
}

}  // namespace bgtq
