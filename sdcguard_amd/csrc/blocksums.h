// Block sums of a matrix of bf16/fp16 outputs, shared by the serving and training checks.
//
// A (row, block) pair is `bs` consecutive outputs of one row (the last block of a row may be narrower, `rem`).
// For each pair the check needs four fp32 sums: plain, signed with the block width's +-1 pattern, of squares and
// of |values| (serve.py:247-254, checksum.py:481-509).  A wave reads 64 consecutive pairs; four lanes share a pair
// in each of four rounds (each reads 4 x 16 bytes of the 256-byte block, in runs of 64 bytes), all sixteen
// loads in flight before any is used, and adds the sums with packed dot products (two elements per instruction)
// and two DPP steps; lane l ends up with pair base + (l & 3) * 16 + (l >> 2).
#pragma once
#include "common.h"

// Where the outputs are: element (batch b, row r, column c) at y[b * sb + r * sm + c * sn].
struct YView {
  const uint16_t* y;
  int64_t sb, sm, sn;
  int64_t m, nb, bs, rem, npairs;      // npairs = batches * m * nb (flat pair index p = (b * m + r) * nb + jb)
  int vec;                             // 16-byte loads (sn == 1; any alignment)
  const float* s_full;                 // +-1 pattern of width bs (a 128-entry row of the sign table)
  const float* s_last;                 // +-1 pattern of width rem
};

// Whether any block is narrower than 128 in a row read in 16-byte pieces
static inline bool blocks_narrow(const YView& v) { return v.vec && (v.rem != 0 || v.bs != 128); }

__device__ __forceinline__ void pair_index(const YView& v, int64_t p, int64_t& b, int64_t& r, int64_t& jb) {
  const uint32_t rr = (uint32_t)p / (uint32_t)v.nb;
  jb = (uint32_t)p - rr * (uint32_t)v.nb;
  b = rr / (uint32_t)v.m;
  r = rr - (uint32_t)b * (uint32_t)v.m;
}

// Division and square root by the hardware's reciprocal and square-root approximations (about 1 ulp): the scores
// only need to agree with the reference's to 1e-3 of the noise, and the special cases keep their IEEE results
// (x / 0 = inf, 0 / 0 = NaN, inf / inf = NaN, sqrt(inf) = inf, sqrt(NaN) = NaN).
__device__ __forceinline__ float fdiv(float a, float b) { return a * __builtin_amdgcn_rcpf(b); }
__device__ __forceinline__ float fsqrt(float a) { return __builtin_amdgcn_sqrtf(a); }

// Four sums of 8 elements (one 16-byte load) with packed dot products: v_dot2_f32_{bf16,f16} adds two products
// to an fp32 accumulator, so each instruction takes two elements: plain sum (x . 1), signed sum (x . s), sum of
// squares (x . x) and sum of |x| (|x| . 1).  `sg2` holds the four sign pairs of these eight columns.
template <int DT>
__device__ __forceinline__ float dot2(uint32_t a, uint32_t b, float c) {
  if constexpr (DT == SDC_BF16) {
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, a), __builtin_bit_cast(bf16x2, b), c, false);
  } else {
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, a), __builtin_bit_cast(f16x2, b), c, false);
  }
}

// a . b + 0, the first term of a sum: the three-operand form takes the zero as an inline constant, where the
// accumulating form (what the compiler picks for dot2(a, b, 0)) needs a register cleared first
template <int DT>
__device__ __forceinline__ float dot2_first(uint32_t a, uint32_t b) {
  float r;
  if constexpr (DT == SDC_BF16) asm("v_dot2_f32_bf16 %0, %1, %2, 0" : "=v"(r) : "v"(a), "v"(b));
  else asm("v_dot2_f32_f16 %0, %1, %2, 0" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

template <int DT>
__device__ __forceinline__ void acc8(u32x4 v, const uint32_t* sg2, float& pl, float& sg, float& sq, float& ab) {
  constexpr uint32_t ONES = DT == SDC_BF16 ? 0x3F803F80u : 0x3C003C00u;
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    pl = dot2<DT>(w[i], ONES, pl);
    sg = dot2<DT>(w[i], sg2[i], sg);
    sq = dot2<DT>(w[i], w[i], sq);
    ab = dot2<DT>(w[i] & 0x7FFF7FFFu, ONES, ab);
  }
}

// 16 bytes at any 2-byte address (global loads take any), read once
typedef u32x4 __attribute__((aligned(2))) u32x4_any;
__device__ __forceinline__ u32x4 load16_any(const uint16_t* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const u32x4_any*>(p));
}

// v's elements moved down by sh (0 .. 8), zeros from the top
__device__ __forceinline__ u32x4 drop_low(u32x4 v, int sh) {
  if (sh & 1) {
    v.x = __builtin_amdgcn_alignbit(v.y, v.x, 16);
    v.y = __builtin_amdgcn_alignbit(v.z, v.y, 16);
    v.z = __builtin_amdgcn_alignbit(v.w, v.z, 16);
    v.w = v.w >> 16;
  }
  if (sh & 2) v = u32x4{v.y, v.z, v.w, 0u};
  if (sh & 4) v = u32x4{v.z, v.w, 0u, 0u};
  if (sh & 8) v = u32x4{0u, 0u, 0u, 0u};
  return v;
}

// The 8 elements at columns c0 .. c0 + 7 of a block of `wid` columns (row: the block's first), zeros past wid: the 16
// bytes are read from the block's last 8 columns back where c0 + 8 passes its end, so nothing past the row is read;
// the block's end must be at least 8 columns from its row's start.
__device__ __forceinline__ u32x4 load8_upto(const uint16_t* row, int c0, int wid) {
  const int off = c0 + 8 <= wid ? c0 : wid - 8, sh = c0 - off;
  const u32x4 v = load16_any(row + off);
  return sh > 0 ? drop_low(v, sh < 8 ? sh : 8) : v;
}

// The signs of 8 columns of a pattern (a table row: zeros past its width) as packed pairs
template <int DT>
__device__ __forceinline__ void pack_signs8(const float* sp, uint32_t* sg2) {
  constexpr uint32_t POS = DT == SDC_BF16 ? 0x3F80u : 0x3C00u, NEG = DT == SDC_BF16 ? 0xBF80u : 0xBC00u;
  const f32x4 s0 = *reinterpret_cast<const f32x4*>(sp), s1 = *reinterpret_cast<const f32x4*>(sp + 4);
  sg2[0] = (s0.x < 0.f ? NEG : POS) | ((s0.y < 0.f ? NEG : POS) << 16);
  sg2[1] = (s0.z < 0.f ? NEG : POS) | ((s0.w < 0.f ? NEG : POS) << 16);
  sg2[2] = (s1.x < 0.f ? NEG : POS) | ((s1.y < 0.f ? NEG : POS) << 16);
  sg2[3] = (s1.z < 0.f ? NEG : POS) | ((s1.w < 0.f ? NEG : POS) << 16);
}

// The four sums of the (row, block) pair each lane keeps: a wave reads 64 consecutive pairs starting at `base`;
// lane l ends up with pair base + (l & 3) * 16 + (l >> 2).  Four lanes share a pair in each of four rounds; all
// sixteen 16-byte loads are issued before any is used (256 bytes per lane in flight).  A block narrower than 128 (a
// row's last) is read the same way, its columns past the end dropped, with its own width's signs (ns2, lane_signs_last).
// Strided rows, and rows of fewer than 8 columns, take an element-wise path.
// NARROW: whether narrower blocks are read so (they cost registers: 4096 x 14336 35 and 42 us without and with them, so
// passes over whole blocks leave them out; blocks_narrow).  In a round that holds a narrower block every lane drops and picks
// its signs (a full block drops nothing); with a path of its own for them such rounds took both, and the signs'
// loads in turn: 96 x 577 x 577, where most rounds do, 39 us, from 41.
template <int DT, bool NARROW>
__device__ __forceinline__ void pair_sums(const YView& a, int64_t base, int lane, const uint32_t* sg2,
                                          const uint32_t* ns2, float& my_pl, float& my_sg, float& my_sq, float& my_ab) {
  const int q = lane & 3;
  int how[4];                           // 0: elements, 1: a full block, 2: a narrower one, 3: a narrower last one
  u32x4 v[4][4];
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const int64_t p = base + g * 16 + (lane >> 2);
    how[g] = 0;
    if (p < a.npairs && a.vec) {
      int64_t b, r, jb;
      pair_index(a, p, b, r, jb);
      if constexpr (!NARROW) {            // (rows read so hold whole blocks only)
        how[g] = 1;
        const uint16_t* yr = a.y + b * a.sb + r * a.sm + jb * 128;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[g][j] = load16_any(yr + 8 * (q + 4 * j));
      } else {
        const bool last = (jb == a.nb - 1) && (a.rem > 0);
        const int wid = (int)(last ? a.rem : a.bs);
        const uint16_t* yr = a.y + b * a.sb + r * a.sm + jb * a.bs;
        if (wid == 128) {
          how[g] = 1;
#pragma unroll
          for (int j = 0; j < 4; ++j) v[g][j] = load16_any(yr + 8 * (q + 4 * j));
        } else if (jb * a.bs + wid >= 8) {
          how[g] = last ? 3 : 2;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int c0 = 8 * (q + 4 * j);
            v[g][j] = load16_any(yr + (c0 + 8 <= wid ? c0 : wid - 8));
          }
        }
      }
    }
  }
  my_pl = my_sg = my_sq = my_ab = 0.f;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const int64_t p = base + g * 16 + (lane >> 2);
    float pl = 0.f, sg = 0.f, sq = 0.f, ab = 0.f;
    auto whole = [&]() {
#pragma unroll
      for (int j = 0; j < 4; ++j) acc8<DT>(v[g][j], &sg2[j * 4], pl, sg, sq, ab);
    };
    auto elements = [&]() {
      int64_t b, r, jb;
      pair_index(a, p, b, r, jb);
      const bool last = (jb == a.nb - 1) && (a.rem > 0);
      const int wid = (int)(last ? a.rem : a.bs);
      const float* sp = last ? a.s_last : a.s_full;
      const uint16_t* yr = a.y + b * a.sb + r * a.sm + jb * a.bs * a.sn;
#pragma unroll 1
      for (int j = 0; j < 4; ++j)
#pragma unroll 1
        for (int e = 0; e < 8; ++e) {
          const int c = 8 * (q + 4 * j) + e;
          if (c < wid) {
            float x = half_to_f32<DT>(yr[c * a.sn]);
            pl += x;
            sg = fmaf(x, sp[c], sg);
            sq = fmaf(x, x, sq);
            ab += fabsf(x);
          }
        }
    };
    if constexpr (!NARROW) {
      if (how[g]) whole();
      else if (p < a.npairs) elements();
    } else {
      if (__builtin_amdgcn_ballot_w64(how[g] >= 2)) {
        if (how[g]) {
          const bool last = how[g] == 3;
          const int wid = last ? (int)a.rem : (int)a.bs;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int sh = 8 * (q + 4 * j) + 8 - wid;
            uint32_t ns[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) ns[e] = last ? ns2[4 * j + e] : sg2[4 * j + e];
            acc8<DT>(drop_low(v[g][j], sh < 0 ? 0 : sh < 8 ? sh : 8), ns, pl, sg, sq, ab);
          }
        }
      } else if (how[g] == 1) {
        whole();
      }
      if (how[g] == 0 && p < a.npairs) elements();
    }
    pl = quad_sum(pl); sg = quad_sum(sg); sq = quad_sum(sq); ab = quad_sum(ab);
    if (q == g) { my_pl = pl; my_sg = sg; my_sq = sq; my_ab = ab; }
  }
}

// The signs of this lane's 32 columns of a full block (chunks q, q+4, q+8, q+12 of 8 columns) as packed pairs; a
// table row holds 128 entries (zeros past its width), so these loads need no bounds test.
template <int DT>
__device__ __forceinline__ void lane_signs(const YView& a, int q, uint32_t* sg2) {
#pragma unroll
  for (int j = 0; j < 4; ++j) pack_signs8<DT>(a.s_full + 8 * (q + 4 * j), &sg2[j * 4]);
}

// The signs of the same columns of the last, narrower block (pair_sums' ns2)
template <int DT>
__device__ __forceinline__ void lane_signs_last(const YView& a, int q, uint32_t* ns2) {
#pragma unroll
  for (int j = 0; j < 4; ++j) pack_signs8<DT>(a.s_last + 8 * (q + 4 * j), &ns2[j * 4]);
}
