// Precise column-block check of C = beta * bias + alpha * (A @ B) with C the fp32 product itself (the accumulator,
// not rounded to 16 bits): checksum.py:537-692 (`matmul_zscores_acc`, `_acc_zscores`, `check_matmul_acc`).
//
// Both sides of every checksum are float64: the block sums of B and of C, and E = A @ B2.  The noise is the fp32
// accumulation's own rounding,
//     u (C1 sqrt(k) |alpha| |a_row|_2 |B_block|_F + (C2 sqrt(k) + C3 k / nfma + sqrt(width)) |C_block|_2),  u = 2^-24,
// judged with the Inf/NaN rules of `_judge_nonfinite` (fp32 outputs, no subnormal step).
// Three launches, no host synchronisation:
//   1. acc_bsums: B2 (fp64 plain and signed block sums of every row of B, in the GEMM's fragment order) and per 64-row
//      slice the partial |B|^2 and max |B| of every block; further workgroups: |a_row|_2 and |a_row|_1 (fp32);
//   2. acc_gemm: E = A @ B2 on the float64 matrix cores, depth split over workgroups (each split its own plane, added
//      by the scorer); further workgroups: |B_block|_F and max |B_block| from the partials, and a bias vector's
//      block sums (fp64) and largest |bias| per block;
//   3. acc_score: one pass over C, 16 lanes per (batch, row, block) for its fp64 plain and signed sums, |C_block|_2
//      and |C_block|_1 (fp32), then a lane per pair scores it; worst keys and the unjudged count go to the result row.
// sdc_matmul_check_acc_stats scores the same check from the block statistics the fused GEMM leaves instead of C
// (fused.py:181-235, `zscores_from_stats`: 2-D, bias vector, alpha = beta = 1; |C_block|_2 is the square root of
// the float64 sum of squares).
#include "blocksums.h"
#include "profile.h"

namespace {

constexpr int SLICE = 64;          // rows of B per acc_bsums workgroup
constexpr int SEG = 32;            // depth of a fragment segment of the GEMM (SLICE is whole segments)
constexpr int MAX_SPLITS = 32;     // depth splits of acc_gemm
constexpr int ACC_WGS = 256;       // workgroups of acc_gemm that fill the chip (one wave per SIMD)
constexpr double ACC_U = 5.9604644775390625e-08;         // 2^-24, checksum.py:558
constexpr double ACC_C1 = 0.6, ACC_C2 = 1.0, ACC_C3 = 1.0;

__device__ __forceinline__ float nan_abs(float v) { return v == v ? fabsf(v) : __builtin_inff(); }

typedef double f64x2 __attribute__((ext_vector_type(2)));
typedef double f64x4 __attribute__((ext_vector_type(4)));

// v's DPP partner's value
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v) {
  return __builtin_bit_cast(double, dpp_i64<CTRL>(__builtin_bit_cast(int64_t, v)));
}
template <int CTRL>
__device__ __forceinline__ float dpp_f32(float v) {
  return __uint_as_float(dpp_u32<CTRL>(__float_as_uint(v)));
}
// sum (maximum) over the 16 lanes of an aligned group (lanes 16 g .. 16 g + 15), in every one of them
__device__ __forceinline__ double sum16_f64(double v) {
  v += dpp_f64<0xB1>(v);
  v += dpp_f64<0x4E>(v);
  v += dpp_f64<0x141>(v);
  v += dpp_f64<0x140>(v);
  return v;
}
__device__ __forceinline__ float sum16_f32(float v) {
  v += dpp_f32<0xB1>(v);
  v += dpp_f32<0x4E>(v);
  v += dpp_f32<0x141>(v);
  v += dpp_f32<0x140>(v);
  return v;
}
__device__ __forceinline__ float max16_f32(float v) {
  v = fmaxf(v, dpp_f32<0xB1>(v));
  v = fmaxf(v, dpp_f32<0x4E>(v));
  v = fmaxf(v, dpp_f32<0x141>(v));
  v = fmaxf(v, dpp_f32<0x140>(v));
  return v;
}
__device__ __forceinline__ double wave_sum_f64(double v) {
  v = sum16_f64(v);
  v += __shfl_xor(v, 16, SDC_WAVE);
  v += __shfl_xor(v, 32, SDC_WAVE);
  return v;
}

struct AccArgs {
  const void* A;                   // (batch_a, m, k) of dtype
  int64_t sab, sam, sak, batch_a;
  const void* B;                   // (batch_b, k, n) of dtype
  int64_t sbb, sbk, sbn, batch_b;
  const float* C;                  // (batch_c, m, n) fp32
  int64_t scb, scm, scn, batch_c;
  int64_t m, k, n, bs, nb, rem, nslice, splits;
  int64_t nseg, nct, segs;         // depth segments of B2, its 16-column tiles, segments per split
  int64_t bwork;                   // acc_bsums' workgroups for B (those past them: row norms)
  int64_t gwork;                   // acc_gemm's workgroups for the product (those past them: block norms)
  int ctg, bmode;                  // groups of column tiles; how acc_bsums reads B (BROWS, BDEPTH, BELEM)
  const void* bias;                // dtype (or fp32 with bias_f32), kind 1: (n), kind 2: (batch, m, n) strides
  int bias_kind, bias_f32;
  int64_t sbias_b, sbias_m, sbias_n;
  double alpha, beta;
  double steps;                    // k / nfma (0: no tensor-core truncation steps)
  float z, abs_floor;
  const float* sign_table;         // 128 x 128, row w - 1 = the pattern of width w
  double* B2T;                     // [batch_b][nseg][nct][4][64][2], see b2_at
  float* part;                     // [batch_b][nslice][nb][2]: sum of squares, max |B|
  float* bstat;                    // [batch_b][nb][2]: |B_block|_F, max |B_block|
  double* bsum;                    // [nb][2]: bias vector block sums (kind 1)
  float* bmax;                     // [nb]: max |bias| of the block (kind 1)
  float* an;                       // [batch_a][2][m]: |a|_2, |a|_1
  double* E;                       // [splits][batch_c][m][2 nb]
  int64_t* result;
  unsigned long long* slots;       // sdc_raise_worst's, cleared by acc_bsums
  float* scores;                   // (batch_c, m, nb, 2) or null
  const double* stats;             // instead of C: (m, nb, 4) plain, signed, squared, absolute block sums of C
  int64_t sst_m, sst_b;            //   (row and block strides, in doubles)
};

__device__ __forceinline__ int64_t bwidth(const AccArgs& a, int64_t jb) {
  return (jb == a.nb - 1 && a.rem > 0) ? a.rem : a.bs;
}

__device__ __forceinline__ float bias_at(const AccArgs& a, int dt, int64_t i) {
  if (a.bias_f32) return reinterpret_cast<const float*>(a.bias)[i];
  const uint16_t w = reinterpret_cast<const uint16_t*>(a.bias)[i];
  return dt == SDC_BF16 ? half_to_f32<SDC_BF16>(w) : half_to_f32<SDC_FP16>(w);
}

// Where B2's value of depth kk and checksum column col is, in the order the GEMM's lanes hold it: lane 16 q + j of the
// fragment of a segment of 32 depths and a tile of 16 columns holds column j, depths 8 q .. 8 q + 7, in four pairs
// (one 16-byte load each, 1 KB a wave).
__device__ __forceinline__ int64_t b2_at(const AccArgs& a, int64_t bb, int64_t kk, int64_t col) {
  const int64_t seg = kk / SEG, q = (kk / 8) % 4, e = kk % 8, lane = 16 * q + col % 16;
  return ((((bb * a.nseg + seg) * a.nct + col / 16) * 4 + e / 2) * 64 + lane) * 2 + e % 2;
}

// ---------------------------------------------------------------------------------------------- 1. B-side sums
// Workgroup (slice of 64 rows of B, block jb, batch bb).  BROWS (row-contiguous B): 16 lanes per row, 8 columns each
// in one 16-byte load at any alignment, 16 rows per pass.  BDEPTH (depth-contiguous B, a weight's transposed view):
// 8 lanes take the slice's 64 depths of a column, 8 each in one 16-byte load, 32 columns per pass; each lane adds its
// depths' sums over its four columns and the 32 lanes of a depth add theirs by DPP, shuffles and LDS.  BELEM: element
// loads.  4096 x 4096 with the row norms of as large an A: 14 us (4.7 TB/s), from 33 + 22 with element loads for all.
// (float64 sums of the bf16/fp16 values, exact up to the sum's size; depths past k read as zeros)
enum { BROWS = 0, BDEPTH = 1, BELEM = 2 };

// |a_row|_2 and |a_row|_1 of four rows, a wave each
template <int DT>
__device__ void acc_anorm(const AccArgs& a, int64_t wg) {
  const int lane = threadIdx.x & 63;
  const int64_t i = wg * 4 + (threadIdx.x >> 6);
  if (i >= a.batch_a * a.m) return;
  const int64_t ba = i / a.m, row = i % a.m;
  const uint16_t* p = reinterpret_cast<const uint16_t*>(a.A) + ba * a.sab + row * a.sam;
  float sq = 0.f, l1 = 0.f;
  auto add = [&](float x) {
    sq = fmaf(x, x, sq);
    l1 += fabsf(x);
  };
  int64_t kk = 0;
  if (a.sak == 1) {
#pragma unroll 4
    for (; kk + 512 <= a.k; kk += 512) {
      const u32x4 v = load16_any(p + kk + 8 * lane);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        add(lo_of<DT>(v[e]));
        add(hi_of<DT>(v[e]));
      }
    }
  }
  for (kk += lane; kk < a.k; kk += 64) add(half_to_f32<DT>(p[kk * a.sak]));
  sq = wave_sum_f32(sq);
  l1 = wave_sum_f32(l1);
  if (lane == 0) {
    a.an[(ba * 2) * a.m + row] = sqrtf(sq);
    a.an[(ba * 2 + 1) * a.m + row] = l1;
  }
}

template <int DT>
__global__ __launch_bounds__(256) void acc_bsums_kernel(AccArgs a) {
  __shared__ float red[4][2];
  __shared__ f64x2 part64[4][SLICE];                // BDEPTH: each wave's plain and signed sums of the slice's depths
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  if (blockIdx.x == 0) sdc_clear_slots(a.slots, 1, t, 256);
  if ((int64_t)blockIdx.x >= a.bwork) return acc_anorm<DT>(a, (int64_t)blockIdx.x - a.bwork);
  const uint32_t wg = blockIdx.x, q = wg / (uint32_t)a.nslice;
  const int64_t sl = wg - q * (uint32_t)a.nslice, jb = q % (uint32_t)a.nb, bb = q / (uint32_t)a.nb;
  const int64_t wid = bwidth(a, jb), kpad = a.nseg * SEG;
  const float* sp = a.sign_table + (wid - 1) * 128;
  const uint16_t* B = reinterpret_cast<const uint16_t*>(a.B) + bb * a.sbb + jb * a.bs * a.sbn;
  float sq = 0.f, mx = 0.f;
  if (a.bmode == BDEPTH) {
    const int o = t & 7, cg = t >> 3;
    const int64_t kk = sl * SLICE + 8 * o;
    const int off = kk + 8 <= a.k ? 0 : (int)(kk - (a.k - 8));       // the last 8 depths, those before kk dropped
    u32x4 v[4];
    float s[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = cg + 32 * i;
      v[i] = load16_any(B + (c < wid ? c : 0) * a.sbn + kk - off);
      s[i] = sp[c];                                                  // (a table row: zeros past its width)
    }
    double pl[8], sg[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) pl[e] = sg[e] = 0.0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      u32x4 x = off > 0 ? drop_low(v[i], off < 8 ? off : 8) : v[i];
      if (cg + 32 * i >= wid) x = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float f = e & 1 ? hi_of<DT>(x[e / 2]) : lo_of<DT>(x[e / 2]);
        pl[e] += (double)f;
        sg[e] += (double)f * (double)s[i];
        sq = fmaf(f, f, sq);
        mx = fmaxf(mx, nan_abs(f));
      }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      // lanes 8 apart hold the same depths: row rotation by 8, then the other rows
      pl[e] += dpp_f64<0x128>(pl[e]);
      sg[e] += dpp_f64<0x128>(sg[e]);
      pl[e] += __shfl_xor(pl[e], 16, SDC_WAVE);
      sg[e] += __shfl_xor(sg[e], 16, SDC_WAVE);
      pl[e] += __shfl_xor(pl[e], 32, SDC_WAVE);
      sg[e] += __shfl_xor(sg[e], 32, SDC_WAVE);
      if (lane < 8) part64[w][8 * o + e] = f64x2{pl[e], sg[e]};
    }
    __syncthreads();
    if (t < SLICE) {
      const int comp = t & 1, pr = t >> 1;                           // a pair of depths of one checksum column
      f64x2 r = {0.0, 0.0};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        r.x += part64[i][2 * pr][comp];
        r.y += part64[i][2 * pr + 1][comp];
      }
      const int64_t k2 = sl * SLICE + 2 * pr;
      if (k2 < kpad) *reinterpret_cast<f64x2*>(a.B2T + b2_at(a, bb, k2, 2 * jb + comp)) = r;
    }
  } else {
    const int c16 = t & 15, r16 = t >> 4;
    // (blocks that end fewer than 8 columns into the row, and any other stride: element loads)
    const bool rows = a.bmode == BROWS && jb * a.bs + wid >= 8;
    u32x4 v[SLICE / 16];
    float s8[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) s8[e] = sp[8 * c16 + e];
    if (rows) {
#pragma unroll
      for (int i = 0; i < SLICE / 16; ++i) {
        const int64_t kk = sl * SLICE + 16 * i + r16;
        v[i] = load8_upto(B + (kk < a.k ? kk : 0) * a.sbk, 8 * c16, (int)wid);
        if (kk >= a.k) v[i] = u32x4{0u, 0u, 0u, 0u};
      }
    }
#pragma unroll
    for (int i = 0; i < SLICE / 16; ++i) {
      const int64_t kk = sl * SLICE + 16 * i + r16;
      double pl = 0.0, sg = 0.0;
      auto add = [&](float x, float sgn) {
        pl += (double)x;
        sg += (double)x * (double)sgn;
        sq = fmaf(x, x, sq);
        mx = fmaxf(mx, nan_abs(x));
      };
      if (rows) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          add(lo_of<DT>(v[i][e]), s8[2 * e]);
          add(hi_of<DT>(v[i][e]), s8[2 * e + 1]);
        }
      } else if (kk < a.k) {
        for (int64_t c = c16; c < wid; c += 16) add(half_to_f32<DT>(B[kk * a.sbk + c * a.sbn]), sp[c]);
      }
      pl = sum16_f64(pl);
      sg = sum16_f64(sg);
      if (c16 < 2 && kk < kpad) a.B2T[b2_at(a, bb, kk, 2 * jb + c16)] = c16 ? sg : pl;
    }
  }
#pragma unroll
  for (int msk = 1; msk < 64; msk <<= 1) {
    sq += __shfl_xor(sq, msk, SDC_WAVE);
    mx = fmaxf(mx, __shfl_xor(mx, msk, SDC_WAVE));
  }
  if (lane == 0) {
    red[w][0] = sq;
    red[w][1] = mx;
  }
  __syncthreads();
  if (t == 0) {
    float sum = red[0][0], m = red[0][1];
    for (int i = 1; i < 4; ++i) {
      sum += red[i][0];
      m = fmaxf(m, red[i][1]);
    }
    float* p = a.part + ((bb * a.nslice + sl) * a.nb + jb) * 2;
    p[0] = sum;
    p[1] = m;
  }
}

// ------------------------------------------------------------------------- 2. block norms and bias block sums
// One wave per (batch of B, block): the slices' partials.  Waves past those: the bias vector's per-block fp64 sums and
// largest |bias| (kind 1).
template <int DT>
__device__ void acc_finish(const AccArgs& a, int64_t wg) {
  const int lane = threadIdx.x & 63;
  const int64_t i = wg * 4 + (threadIdx.x >> 6);
  const int64_t nbb = a.batch_b * a.nb;
  if (i < nbb) {
    const int64_t bb = i / a.nb, jb = i % a.nb;
    float s = 0.f, m = 0.f;
    for (int64_t sl = lane; sl < a.nslice; sl += 64) {
      const float* p = a.part + ((bb * a.nslice + sl) * a.nb + jb) * 2;
      s += p[0];
      m = fmaxf(m, p[1]);
    }
    s = wave_sum_f32_dpp(s);
    m = wave_max_f32_dpp(m);
    if (lane == 0) {
      a.bstat[i * 2] = sqrtf(s);
      a.bstat[i * 2 + 1] = m;
    }
  } else if (a.bias_kind == 1 && i < nbb + a.nb) {
    const int64_t jb = i - nbb, wid = bwidth(a, jb);
    const float* sp = a.sign_table + (wid - 1) * 128;
    double pl = 0.0, sg = 0.0;
    float mx = 0.f;
    for (int64_t c = lane; c < wid; c += 64) {
      const float v = bias_at(a, DT, (jb * a.bs + c) * a.sbias_n);
      pl += (double)v;
      sg += (double)v * (double)sp[c];
      mx = fmaxf(mx, nan_abs(v));
    }
    pl = wave_sum_f64(pl);
    sg = wave_sum_f64(sg);
    mx = wave_max_f32_dpp(mx);
    if (lane == 0) {
      a.bsum[jb * 2] = pl;
      a.bsum[jb * 2 + 1] = sg;
      a.bmax[jb] = mx;
    }
  }
}

// ------------------------------------------------------------------------------------- 3. E = A @ B2 (float64)
// v_mfma_f64_16x16x4_f64: lane 16 q + j holds A[row j][depth q] and B[depth q][column j]; register r of the result is
// row 4 r + q, column j.  Which depths four lanes' values stand for is free as long as A and B agree, so lane group q
// takes depths 8 q .. 8 q + 7 of a segment of 32: one 16-byte load of A per row tile, four of B2 (in that order in
// memory) per column tile, eight steps.  A wave owns 32 rows x NCT column tiles and one part of the depth; the four waves of
// a workgroup are 128 rows of the same part, so they share B2 in the L1.  The next segment's loads are issued before
// a segment's products (at NCT = 4, 64 of them of 64 clocks each), which hides them with one wave per SIMD.  Bound by the float64
// matrix rate: 2.1 GFLOP of 4096 x 64 x 4096 take 48 us (45 of 78.6 TFLOP/s; 195 us as a tiled VALU GEMM through LDS).
// VEC: A's rows are depth-contiguous and at least 8 long (16-byte loads at any alignment; depths past the end are
// dropped); otherwise element loads.
template <int DT, int NCT, bool VEC>
__global__ __launch_bounds__(256) void acc_gemm_kernel(AccArgs a) {
  const int t = threadIdx.x, lane = t & 63, w = t >> 6, j = lane & 15, q = lane >> 4;
  if ((int64_t)blockIdx.x >= a.gwork) return acc_finish<DT>(a, (int64_t)blockIdx.x - a.gwork);
  // (depth parts fastest: with a multiple of eight of them an XCD's workgroups read the same part of B2)
  const int64_t nrt = sdc_cdiv(a.m, 128);
  const int64_t split = blockIdx.x % a.splits, r1 = blockIdx.x / a.splits;
  const int64_t cgp = r1 % a.ctg, r2 = r1 / a.ctg;
  const int64_t rt = r2 % nrt, bc = r2 / nrt;
  const int64_t ba = a.batch_a == 1 ? 0 : bc, bb = a.batch_b == 1 ? 0 : bc;
  const int64_t r0 = rt * 128 + 32 * w;
  if (r0 >= a.m) return;
  const int64_t s0 = split * a.segs, s1 = s0 + a.segs < a.nseg ? s0 + a.segs : a.nseg;
  const uint16_t* ap[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int64_t row = r0 + 16 * i + j;
    ap[i] = reinterpret_cast<const uint16_t*>(a.A) + ba * a.sab + (row < a.m ? row : a.m - 1) * a.sam;
  }
  const f64x2* bp[NCT];
#pragma unroll
  for (int c = 0; c < NCT; ++c) {
    const int64_t ct = cgp * NCT + c < a.nct ? cgp * NCT + c : a.nct - 1;
    bp[c] = reinterpret_cast<const f64x2*>(a.B2T) + (bb * a.nseg * a.nct + ct) * 256 + lane;
  }
  f64x4 acc[2][NCT];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int c = 0; c < NCT; ++c) acc[i][c] = f64x4{0.0, 0.0, 0.0, 0.0};
  struct Frag {
    u32x4 a[2];
    f64x2 b[NCT][4];
  };
  auto load = [&](Frag& f, int64_t sg) {
    const int64_t kk = SEG * sg + 8 * q;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if constexpr (VEC) {
        f.a[i] = load16_any(ap[i] + (kk + 8 <= a.k ? kk : a.k - 8));
      } else {
        uint16_t e[8];
#pragma unroll
        for (int x = 0; x < 8; ++x) e[x] = ap[i][(kk + x < a.k ? kk + x : a.k - 1) * a.sak];
#pragma unroll
        for (int x = 0; x < 4; ++x) f.a[i][x] = e[2 * x] | ((uint32_t)e[2 * x + 1] << 16);
      }
    }
#pragma unroll
    for (int c = 0; c < NCT; ++c)
#pragma unroll
      for (int p = 0; p < 4; ++p) f.b[c][p] = bp[c][sg * a.nct * 256 + 64 * p];
  };
  auto product = [&](Frag& f, int64_t sg) {
    const int64_t kk = SEG * sg + 8 * q;
    if (SEG * (sg + 1) > a.k) {                       // the last segment: depths past the end as zeros
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        if constexpr (VEC) {
          const int64_t off = kk + 8 - a.k;
          f.a[i] = off > 0 ? drop_low(f.a[i], off < 8 ? (int)off : 8) : f.a[i];
        } else {
#pragma unroll
          for (int x = 0; x < 4; ++x)
            f.a[i][x] &= (kk + 2 * x < a.k ? 0xFFFFu : 0u) | (kk + 2 * x + 1 < a.k ? 0xFFFF0000u : 0u);
        }
      }
    }
#pragma unroll
    for (int p = 0; p < 4; ++p)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        double av[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) av[i] = (double)(h ? hi_of<DT>(f.a[i][p]) : lo_of<DT>(f.a[i][p]));
#pragma unroll
        for (int c = 0; c < NCT; ++c)
#pragma unroll
          for (int i = 0; i < 2; ++i)
            acc[i][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[i], f.b[c][p][h], acc[i][c], 0, 0, 0);
      }
  };
  if (s0 < s1) {
    Frag fx, fy;
    const int64_t last = s1 - 1;
    load(fx, s0);
    for (int64_t sg = s0; sg < s1; sg += 2) {
      load(fy, sg + 1 < last ? sg + 1 : last);        // (past the last: the last once more, unused)
      __builtin_amdgcn_sched_barrier(0);
      product(fx, sg);
      if (sg + 1 >= s1) break;
      load(fx, sg + 2 < last ? sg + 2 : last);
      __builtin_amdgcn_sched_barrier(0);
      product(fy, sg + 1);
    }
  }
  const int64_t nc = 2 * a.nb;
  double* Ep = a.E + ((split * a.batch_c + bc) * a.m) * nc;
#pragma unroll
  for (int c = 0; c < NCT; ++c) {
    const int64_t col = (cgp * NCT + c) * 16 + j;
    if (col >= nc) continue;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t row = r0 + 16 * i + 4 * r + q;
        if (row < a.m) Ep[row * nc + col] = acc[i][c][r];
      }
  }
}

// ------------------------------------------------------------------------------------------------ 4. scoring
// One checksum of the precise check, scored as checksum.py:640-670 scores it: z = |expected - actual| / (noise +
// abs_floor) in float64 (the plain one also against the L1 bound), then `_judge_nonfinite` with fp32 outputs.
__device__ __forceinline__ float acc_judge(double e, double act, float noise, float worst, float bound, float cn,
                                           float wf, bool plain, const AccArgs& a, float& den32) {
  const float inf = __builtin_inff();
  const float den = noise + a.abs_floor;
  den32 = den;
  const double diff = fabs(e - act);
  double zd = diff / (double)den;
  if (plain) {
    const double zw = diff / (double)worst * (double)a.z;
    zd = (zd == zd && zw == zw) ? fmin(zd, zw) : __builtin_nan("");
  }
  float zf = (float)zd;
  const bool e_bad = !(fabs(e) < __builtin_inf());
  const bool a_bad = !(fabs(act) < __builtin_inf()) && !e_bad;
  const bool big = !(noise < inf) && !e_bad && !a_bad;
  const float lim = bound * 1.01f;
  zf = zf == zf ? zf : -1.f;
  zf = e_bad ? -1.f : zf;
  const float cap = bound * (float)(1.02 + (double)a.k * 2.384185791015625e-07);
  const bool imposs = !e_bad && !a_bad && !big && (lim < 1e18f) && (cn > cap * sqrtf(wf));
  zf = imposs ? inf : zf;
  zf = a_bad ? (lim < 1e18f ? inf : -1.f) : zf;
  zf = big ? (lim < 1e18f ? inf : -1.f) : zf;
  return zf;
}

// 128 pairs per workgroup, 32 per wave: in eight rounds lanes 16 g .. 16 g + 15 take one (batch, row, block) pair each,
// lane c16 the columns 8 c16 .. 8 c16 + 7 of a full 128-wide block of a row-contiguous C (two 16-byte loads, those of
// all rounds issued first) or c16, c16 + 16, ... of any other; the sums go to LDS and then 128 lanes score a pair each
// (scoring, some 600 instructions in float64, cost more than the pass with one lane of 16 at it: 4096 x 4096 51 us,
// now 21).
constexpr int SPAIRS = 128;
typedef f32x4 __attribute__((aligned(4))) f32x4_any;

template <int DT>
__global__ __launch_bounds__(256) void acc_score_kernel(AccArgs a) {
  __shared__ double ssum[4][SPAIRS];          // plain and signed sums of C, of the bias matrix
  __shared__ float fsum[3][SPAIRS];           // |C_block|_2^2, |C_block|_1, max |bias|
  __shared__ int64_t rk[2], rd[2];
  __shared__ int ru[2];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6, c16 = t & 15;
  const int64_t npairs = a.batch_c * a.m * a.nb;
  const int64_t p0 = (int64_t)blockIdx.x * SPAIRS;
  const uint32_t nb = (uint32_t)a.nb, m = (uint32_t)a.m;      // (pair indexes fit 32 bits)
  // the row's keys so far (keys only grow)
  const int64_t seen0 = __atomic_load_n(a.result, __ATOMIC_RELAXED);
  const int64_t seen1 = __atomic_load_n(a.result + 1, __ATOMIC_RELAXED);
  if (!a.stats) {
    constexpr int NR = SPAIRS / 16;
    auto pair_at = [&](int r) { return 32 * w + 4 * r + (lane >> 4); };
    auto where = [&](uint32_t p, int64_t& jb, int64_t& row, int64_t& bc) {
      const uint32_t q = p / nb;
      jb = p - q * nb;
      bc = q / m;
      row = q - (uint32_t)bc * m;
    };
    f32x4 v[NR][2];
    bool fast[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const int64_t p = p0 + pair_at(r);
      fast[r] = false;
      if (p < npairs && a.scn == 1) {
        int64_t jb, row, bc;
        where((uint32_t)p, jb, row, bc);
        if (bwidth(a, jb) == 128) {
          fast[r] = true;
          const float* cp = a.C + bc * a.scb + row * a.scm + jb * a.bs + 8 * c16;
          v[r][0] = __builtin_nontemporal_load(reinterpret_cast<const f32x4_any*>(cp));
          v[r][1] = __builtin_nontemporal_load(reinterpret_cast<const f32x4_any*>(cp + 4));
        }
      }
    }
    float s8[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) s8[e] = a.sign_table[(a.bs - 1) * 128 + 8 * c16 + e];
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const int at = pair_at(r);
      const int64_t p = p0 + at;
      double pl = 0.0, sg = 0.0, bpl = 0.0, bsg = 0.0;
      float sq = 0.f, l1 = 0.f, bmx = 0.f;
      if (fast[r]) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float x = v[r][e / 4][e % 4];
          pl += (double)x;
          sg += (double)x * (double)s8[e];
          sq = fmaf(x, x, sq);
          l1 += fabsf(x);
        }
      }
      if (p < npairs && (!fast[r] || a.bias_kind == 2)) {
        int64_t jb, row, bc;
        where((uint32_t)p, jb, row, bc);
        const int64_t wid = bwidth(a, jb);
        const float* sp = a.sign_table + (wid - 1) * 128;
        if (!fast[r]) {
          const int64_t cbase = bc * a.scb + row * a.scm + jb * a.bs * a.scn;
          for (int64_t c = c16; c < wid; c += 16) {
            const float x = a.C[cbase + c * a.scn];
            pl += (double)x;
            sg += (double)x * (double)sp[c];
            sq = fmaf(x, x, sq);
            l1 += fabsf(x);
          }
        }
        if (a.bias_kind == 2) {
          const int64_t bb0 = bc * a.sbias_b + row * a.sbias_m + jb * a.bs * a.sbias_n;
          for (int64_t c = c16; c < wid; c += 16) {
            const float x = bias_at(a, DT, bb0 + c * a.sbias_n);
            bpl += (double)x;
            bsg += (double)x * (double)sp[c];
            bmx = fmaxf(bmx, nan_abs(x));
          }
        }
      }
      pl = sum16_f64(pl);
      sg = sum16_f64(sg);
      sq = sum16_f32(sq);
      l1 = sum16_f32(l1);
      if (a.bias_kind == 2) {
        bpl = sum16_f64(bpl);
        bsg = sum16_f64(bsg);
        bmx = max16_f32(bmx);
      }
      if (c16 == 0) {
        ssum[0][at] = pl;
        ssum[1][at] = sg;
        ssum[2][at] = bpl;
        ssum[3][at] = bsg;
        fsum[0][at] = sq;
        fsum[1][at] = l1;
        fsum[2][at] = bmx;
      }
    }
    __syncthreads();
  }
  if (t < SPAIRS) {                                   // (whole waves: two of the four)
    int64_t key = 0, keyd = 0;
    int unk = 0;
    const int64_t p = p0 + t;
    if (p < npairs) {
      const uint32_t q = (uint32_t)p / nb;
      const int64_t jb = (uint32_t)p - q * nb, bc = q / m, row = q - (uint32_t)bc * m;
      const int64_t wid = bwidth(a, jb);
      double pl, sg, bpl = 0.0, bsg = 0.0, sqd = 0.0;
      float sq = 0.f, l1, bmx = 0.f;
      if (a.stats) {                                  // the fused kernel's block statistics (fused.py:205-207)
        const double* st = a.stats + row * a.sst_m + jb * a.sst_b;
        pl = st[0];
        sg = st[1];
        sqd = st[2];
        l1 = (float)st[3];
      } else {
        pl = ssum[0][t];
        sg = ssum[1][t];
        bpl = ssum[2][t];
        bsg = ssum[3][t];
        sq = fsum[0][t];
        l1 = fsum[1][t];
        bmx = fsum[2][t];
      }
      const int64_t ba = a.batch_a == 1 ? 0 : bc, bb = a.batch_b == 1 ? 0 : bc;
      const int64_t nc = 2 * a.nb;
      double e0 = 0.0, e1 = 0.0;
#pragma unroll 4
      for (int64_t s = 0; s < a.splits; ++s) {
        const f64x2 ev = *reinterpret_cast<const f64x2*>(a.E + ((s * a.batch_c + bc) * a.m + row) * nc + 2 * jb);
        e0 += ev.x;
        e1 += ev.y;
      }
      const float anorm = a.an[(ba * 2) * a.m + row], al1 = a.an[(ba * 2 + 1) * a.m + row];
      const float bfrob = a.bstat[(bb * a.nb + jb) * 2], bmaxb = a.bstat[(bb * a.nb + jb) * 2 + 1];
      float bound = al1 * bmaxb;
      if (a.alpha != 1.0) {
        e0 *= a.alpha;
        e1 *= a.alpha;
        bound = bound * (float)fabs(a.alpha);
      }
      if (a.bias_kind != 0 && a.beta != 0.0) {
        if (a.bias_kind == 1) {
          bpl = a.bsum[jb * 2];
          bsg = a.bsum[jb * 2 + 1];
          bmx = a.bmax[jb];
        }
        e0 += a.beta * bpl;
        e1 += a.beta * bsg;
        bound = bound + (float)fabs(a.beta) * bmx;
      }
      const float wf = (float)wid;
      // from statistics: sqrt of the float64 sum of squares (a NaN stays NaN), rounded to fp32
      const float cn = a.stats ? (float)sqrt(sqd < 0.0 ? 0.0 : sqd) : sqrtf(sq);
      const float per_out_u = (float)((ACC_C2 * sqrt((double)a.k) + ACC_C3 * a.steps + sqrt((double)wid)) * ACC_U);
      float prod = (anorm * bfrob) * (float)(ACC_C1 * sqrt((double)a.k) * fabs(a.alpha) * ACC_U);
      prod = fabsf(prod) < __builtin_inff() ? prod : bound * (float)(ACC_U * 128.0);
      const float noise = cn * per_out_u + prod;
      const float worst = (l1 * per_out_u + prod) + a.abs_floor;
      float d0, d1;
      const float z0 = acc_judge(e0, pl, noise, worst, bound, cn, wf, true, a, d0);
      const float z1 = acc_judge(e1, sg, noise, worst, bound, cn, wf, false, a, d1);
      const int64_t flat = ((bc * a.m + row) * a.nb + jb);
      if (a.scores) {
        a.scores[2 * flat] = z0;
        a.scores[2 * flat + 1] = z1;
      }
      unk = (z0 < 0.f) + (z1 < 0.f);
      const bool sec = z1 > z0;
      const float zc = sec ? z1 : z0, dc = sec ? d1 : d0;
      const int64_t zb = fbits64(fmaxf(zc, 0.f));
      key = (zb << 32) | ((flat * 2 + (sec ? 1 : 0)) & 0xFFFFFFFFll);
      keyd = (zb << 32) | (fbits64(dc) & 0xFFFFFFFFll);
    }
    key = wave_max_i64_dpp(key);
    keyd = wave_max_i64_dpp(keyd);
    unk = wave_sum_i32_dpp(unk);
    if (lane == 0) {
      rk[w] = key;
      rd[w] = keyd;
      ru[w] = unk;
    }
  }
  __syncthreads();
  if (t == 0) {
    const int64_t k0 = rk[0] > rk[1] ? rk[0] : rk[1], d0 = rd[0] > rd[1] ? rd[0] : rd[1];
    const int u = ru[0] + ru[1];
    sdc_raise_worst(a.result, a.slots, k0, d0, seen0, seen1);
    if (u > 0) atomicAdd((unsigned long long*)(a.result + 2), (unsigned long long)u);
  }
}

struct AccLayout {
  int64_t nb, nslice, nseg, nct, splits, segs;
  int ctg, tiles;                  // groups of column tiles, tiles a group (1 .. 4)
  int64_t off_b2, off_part, off_bstat, off_bsum, off_bmax, off_an, off_slots, off_e, total;   // bytes
};

AccLayout acc_layout(int64_t batch_a, int64_t batch_b, int64_t batch_c, int64_t m, int64_t k, int64_t n,
                     int64_t bs) {
  AccLayout L{};
  L.nb = sdc_cdiv(n, bs);
  L.nslice = sdc_cdiv(k, SLICE);
  L.nseg = sdc_cdiv(k, SEG);
  L.nct = sdc_cdiv(2 * L.nb, 16);
  L.ctg = (int)sdc_cdiv(L.nct, 4);
  L.tiles = (int)sdc_cdiv(L.nct, L.ctg);
  // depth parts until the chip is full, each at least two segments deep; whole eights of them where there are as many
  const int64_t wgs = sdc_cdiv(m, 128) * L.ctg * batch_c;
  int64_t s = sdc_cdiv(ACC_WGS, wgs);
  const int64_t smax = L.nseg / 2 > 1 ? L.nseg / 2 : 1;
  s = s < smax ? s : smax;
  s = s < MAX_SPLITS ? s : MAX_SPLITS;
  s = s >= 8 ? s / 8 * 8 : s;
  L.segs = sdc_cdiv(L.nseg, s);
  L.splits = sdc_cdiv(L.nseg, L.segs);
  auto al = [](int64_t x) { return (x + 255) / 256 * 256; };
  int64_t o = 0;
  L.off_b2 = o; o += al(batch_b * L.nseg * L.nct * 512 * 8);
  L.off_part = o; o += al(batch_b * L.nslice * L.nb * 2 * 4);
  L.off_bstat = o; o += al(batch_b * L.nb * 2 * 4);
  L.off_bsum = o; o += al(L.nb * 2 * 8);
  L.off_bmax = o; o += al(L.nb * 4);
  L.off_an = o; o += al(batch_a * 2 * m * 4);
  L.off_slots = o; o += al(SDC_SLOT_FLOATS * 4);
  L.off_e = o; o += al(L.splits * batch_c * m * 2 * L.nb * 8);
  L.total = o;
  return L;
}

template <int DT, bool VEC>
void acc_gemm_launch(const AccArgs& a, int tiles, dim3 grid, hipStream_t stream) {
  if (tiles == 1) hipLaunchKernelGGL((acc_gemm_kernel<DT, 1, VEC>), grid, dim3(256), 0, stream, a);
  else if (tiles == 2) hipLaunchKernelGGL((acc_gemm_kernel<DT, 2, VEC>), grid, dim3(256), 0, stream, a);
  else if (tiles == 3) hipLaunchKernelGGL((acc_gemm_kernel<DT, 3, VEC>), grid, dim3(256), 0, stream, a);
  else hipLaunchKernelGGL((acc_gemm_kernel<DT, 4, VEC>), grid, dim3(256), 0, stream, a);
}

// (the sizes, operands, bias, scale and workspace pointer `ws` of `a` are the caller's)
template <int DT>
int acc_run(AccArgs a, const AccLayout& L, uint8_t* ws, hipStream_t stream) {
  a.nb = L.nb; a.nslice = L.nslice; a.nseg = L.nseg; a.nct = L.nct; a.ctg = L.ctg; a.splits = L.splits; a.segs = L.segs;
  a.B2T = (double*)(ws + L.off_b2); a.part = (float*)(ws + L.off_part); a.bstat = (float*)(ws + L.off_bstat);
  a.bsum = (double*)(ws + L.off_bsum); a.bmax = (float*)(ws + L.off_bmax); a.an = (float*)(ws + L.off_an);
  a.E = (double*)(ws + L.off_e);
  // 16-byte loads of 8 elements need 8 of them to be there: rows of at least 8 columns, columns of at least 8 depths
  a.bmode = a.sbn == 1 && a.n >= 8 ? BROWS : a.sbk == 1 && a.k >= 8 ? BDEPTH : BELEM;
  a.bwork = L.nslice * L.nb * a.batch_b;
  a.gwork = sdc_cdiv(a.m, 128) * L.ctg * L.splits * a.batch_c;
  const int64_t pgrid = sdc_cdiv(a.batch_c * a.m * L.nb, SPAIRS);
  a.slots = sdc_slots_for(pgrid, (unsigned long long*)(ws + L.off_slots));
  const int64_t bgrid = a.bwork + sdc_cdiv(a.batch_a * a.m, 4), ggrid = a.gwork + sdc_cdiv(a.batch_b * L.nb + L.nb, 4);
  if (bgrid > 0x7FFFFFFFll || ggrid > 0x7FFFFFFFll) return SDC_EUNSUPPORTED;
  {
    SdcProf prof("acc_bsums", stream);
    hipLaunchKernelGGL(acc_bsums_kernel<DT>, dim3((unsigned)bgrid), dim3(256), 0, stream, a);
    SDC_LAUNCH_CHECK();
  }
  {
    SdcProf prof("acc_gemm", stream);
    if (a.sak == 1 && a.k >= 8) acc_gemm_launch<DT, true>(a, L.tiles, dim3((unsigned)ggrid), stream);
    else acc_gemm_launch<DT, false>(a, L.tiles, dim3((unsigned)ggrid), stream);
    SDC_LAUNCH_CHECK();
  }
  {
    SdcProf prof("acc_score", stream);
    hipLaunchKernelGGL(acc_score_kernel<DT>, dim3((unsigned)pgrid), dim3(256), 0, stream, a);
    SDC_LAUNCH_CHECK();
  }
  return SDC_OK;
}

}  // namespace

extern "C" int64_t sdc_matmul_check_acc_workspace(int64_t batch_a, int64_t batch_b, int64_t batch_c, int64_t m,
                                                  int64_t k, int64_t n, int64_t bs) {
  if (batch_a < 1 || batch_b < 1 || batch_c < 1 || m < 1 || k < 1 || n < 1 || bs < 1) return 0;
  return acc_layout(batch_a, batch_b, batch_c, m, k, n, bs < 128 ? bs : 128).total + 256;
}

extern "C" int sdc_matmul_check_acc_stats(int dtype, const void* A, int64_t sam, int64_t sak, const void* B,
                                          int64_t sbk, int64_t sbn, const double* stats, int64_t sst_m,
                                          int64_t sst_b, int64_t m, int64_t k, int64_t n, const void* bias,
                                          int bias_f32, float nfma, float z, float abs_floor,
                                          const float* sign_table, int64_t* result, void* workspace,
                                          int64_t workspace_bytes, float* scores_out, hipStream_t stream) {
  SDC_CLEAR_ERRORS();
  if (dtype != SDC_BF16 && dtype != SDC_FP16) return SDC_EUNSUPPORTED;
  if (!A || !B || !stats || !sign_table || !result) return SDC_EINVAL;
  if (m < 1 || k < 1 || n < 1) return SDC_EINVAL;
  const int64_t bw = n < 128 ? n : 128;
  const AccLayout L = acc_layout(1, 1, 1, m, k, n, bw);
  if (m * L.nb * 2 > 0xFFFFFFFFll) return SDC_EUNSUPPORTED;
  if (!workspace || workspace_bytes < L.total + 256) return SDC_EWORKSPACE;
  uint8_t* ws = (uint8_t*)(((uintptr_t)workspace + 255) & ~(uintptr_t)255);
  AccArgs a{};
  a.A = A; a.sab = 0; a.sam = sam; a.sak = sak; a.batch_a = 1;
  a.B = B; a.sbb = 0; a.sbk = sbk; a.sbn = sbn; a.batch_b = 1;
  a.C = nullptr; a.batch_c = 1;
  a.stats = stats; a.sst_m = sst_m; a.sst_b = sst_b;
  a.m = m; a.k = k; a.n = n; a.bs = bw; a.rem = n % bw;
  a.bias = bias; a.bias_kind = bias ? 1 : 0; a.bias_f32 = bias_f32; a.sbias_n = 1;
  a.alpha = 1.0; a.beta = 1.0; a.steps = nfma > 0.f ? (double)k / (double)nfma : 0.0;
  a.z = z; a.abs_floor = abs_floor; a.sign_table = sign_table;
  a.result = result; a.scores = scores_out;
  return dtype == SDC_BF16 ? acc_run<SDC_BF16>(a, L, ws, stream) : acc_run<SDC_FP16>(a, L, ws, stream);
}

extern "C" int sdc_matmul_check_acc(int dtype, const void* A, int64_t sab, int64_t sam, int64_t sak, int64_t batch_a,
                                    const void* B, int64_t sbb, int64_t sbk, int64_t sbn, int64_t batch_b,
                                    const float* C, int64_t scb, int64_t scm, int64_t scn, int64_t batch_c, int64_t m,
                                    int64_t k, int64_t n, int64_t bs, const void* bias, int bias_kind, int64_t sbias_b,
                                    int64_t sbias_m, int64_t sbias_n, float alpha, float beta, float nfma, float z,
                                    float abs_floor, const float* sign_table, int64_t* result, void* workspace,
                                    int64_t workspace_bytes, float* scores_out, hipStream_t stream) {
  SDC_CLEAR_ERRORS();
  if (dtype != SDC_BF16 && dtype != SDC_FP16) return SDC_EUNSUPPORTED;
  if (!A || !B || !C || !sign_table || !result) return SDC_EINVAL;
  if (m < 1 || k < 1 || n < 1 || bs < 1 || bs > 128) return SDC_EINVAL;
  if (batch_c < 1 || (batch_a != 1 && batch_a != batch_c) || (batch_b != 1 && batch_b != batch_c)) return SDC_EINVAL;
  const int kind = bias_kind & 3, bias32 = (bias_kind & 4) != 0;
  if (kind > 2 || (kind && !bias)) return SDC_EINVAL;
  const int64_t bw = bs < n ? bs : n;
  const AccLayout L = acc_layout(batch_a, batch_b, batch_c, m, k, n, bw);
  if (m * L.nb * batch_c * 2 > 0xFFFFFFFFll) return SDC_EUNSUPPORTED;      // flat indexes fit the key's 32 bits
  if (!workspace || workspace_bytes < L.total + 256) return SDC_EWORKSPACE;
  uint8_t* ws = (uint8_t*)(((uintptr_t)workspace + 255) & ~(uintptr_t)255);
  AccArgs a{};
  a.A = A; a.sab = sab; a.sam = sam; a.sak = sak; a.batch_a = batch_a;
  a.B = B; a.sbb = sbb; a.sbk = sbk; a.sbn = sbn; a.batch_b = batch_b;
  a.C = C; a.scb = scb; a.scm = scm; a.scn = scn; a.batch_c = batch_c;
  a.m = m; a.k = k; a.n = n; a.bs = bw; a.rem = n % bw;
  a.bias = bias; a.bias_kind = kind; a.bias_f32 = bias32; a.sbias_b = sbias_b; a.sbias_m = sbias_m; a.sbias_n = sbias_n;
  a.alpha = alpha; a.beta = beta; a.steps = nfma > 0.f ? (double)k / (double)nfma : 0.0;
  a.z = z; a.abs_floor = abs_floor; a.sign_table = sign_table;
  a.result = result; a.scores = scores_out;
  return dtype == SDC_BF16 ? acc_run<SDC_BF16>(a, L, ws, stream) : acc_run<SDC_FP16>(a, L, ws, stream);
}
