// Expected side E = A @ (three parts of the block sums) for an A that the whole-line GEMMs cannot stream: rows that are
// contiguous across each other (a weight gradient's dy^T: element (row, kk) at A[kk * sak + row]), or rows whose
// starts are not 16-byte aligned or whose depth is not whole 64s (an output head of 50257 columns).
//
// As in the tall-tile GEMM, a workgroup of 4 waves owns a 128 x 64 tile of E (128 x 32 for at most 32 columns: half the
// products, and two workgroups a CU) over one depth part, each wave a share of that part's 64-deep segments, and the
// parts of B come in fragment order (zero past the depth); the waves' sums meet in LDS at the end.  A, by MODE:
//   ROWS (rows contiguous): straight into the MFMA operands' registers, four 16-deep steps ahead.  Lane (r, h) reads rows
//     4 r .. 4 r + 3 (8 bytes) at the eight depths 32 h + 8 j .. + 7 of step j, 256 contiguous bytes an instruction and
//     half wave; four v_perm pairs per row turn the eight depths x four rows into four fragments, fragment i holding
//     rows 4 r + i (which rows a fragment holds is free: the epilogue knows).  (Loads off a word boundary run at three
//     quarters of the rate; 12 bytes from the word below, shifted, cost the registers of the second workgroup.)
//   DEPTH (depth contiguous): the next segment's 128 rows x 128 bytes in coalesced 16-byte loads at any alignment, 8
//     rows an instruction, then through the wave's own 16 KB of LDS (16-byte piece p of row r at position p ^ (r % 8)).
//     Loads of a row a lane touched 64 lines an instruction, each line again by seven more.
// Bound by the loads in flight (16 KB a wave) and the matrix cores.  Measured on MI355X: dy^T 14336 x 4096 (64 columns)
// 34-36 us, from 125 us with the staged GEMM's element loads; with 12 columns, dy 1024 x 50257 37 us (from 66 us with loads
// straight into the operands' registers and 64-column tiles) and dy^T 50257 x 1024 40 us (from 69 us, with
// every row tile's last segment element by element).
#include "blocksums.h"
#include "common.h"
#include "gemm.h"
#include "mfma_pipe.h"
#include "profile.h"
#include "split.h"

namespace {

constexpr int NW = 4, TRF = 4, TR = 128, RP = TR + 4;
enum { DEPTH = 0, ROWS = 1 };

typedef u32x2 __attribute__((aligned(2))) u32x2_any;        // 8 and 16 bytes at any 2-byte address
typedef u32x4 __attribute__((aligned(2))) u32x4_lane;

// Which element of a 128 x 32 TCF tile lane l of wave w stores at step s of the row-major epilogue: columns col .. + 3 of
// row `row`.  Every column it reads from LDS has to be one of the tile's own: the waves' sums are a tile after the other
// there, and nothing follows the last.
template <int TCF>
struct RowMajor {
  static constexpr int TC = 32 * TCF, LANES = TC / 4, ROWS_PER = 64 / LANES, STEPS = TR / (ROWS_PER * NW);
  static constexpr int col(int l) { return 4 * (l % LANES); }
  static constexpr int row(int w, int s, int l) { return w * (TR / NW) + ROWS_PER * s + l / LANES; }
  // every element of the tile once, none outside it
  static constexpr bool covers_tile() {
    bool seen[TR * TC / 4] = {};
    for (int w = 0; w < NW; ++w)
      for (int s = 0; s < STEPS; ++s)
        for (int l = 0; l < 64; ++l) {
          const int r = row(w, s, l), c = col(l);
          if (r < 0 || r >= TR || c < 0 || c + 4 > TC || seen[(r * TC + c) / 4]) return false;
          seen[(r * TC + c) / 4] = true;
        }
    for (bool b : seen)
      if (!b) return false;
    return true;
  }
};
static_assert(RowMajor<1>::covers_tile() && RowMajor<2>::covers_tile(), "the row-major epilogue stays in the tile's sums");

// MODE: ROWS needs g.sam 1, g.sak >= g.m >= 4; DEPTH needs g.sak 1.  TCF: 32-column fragments of the tile
template <int DT, int MODE, int TCF>
__global__ __launch_bounds__(64 * NW, TCF == 1 ? 2 : 1) void lane_gemm_kernel(GemmArgs g) {
  constexpr int TC = 32 * TCF;
  static_assert(NW * TC * RP * 4 >= NW * TR * 128, "DEPTH: the waves' segments fit the epilogue's LDS");
  __shared__ __attribute__((aligned(16))) float red[NW * TC * RP];
  __shared__ float xred[NW][TR][2];
  const int t = threadIdx.x, lane = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int r = lane & 31, h = lane >> 5;
  const int64_t m = g.m, k = g.k, N = g.N;
  const uint32_t nct = ((uint32_t)N + TC - 1) / TC, ncf = ((uint32_t)N + 31) / 32;
  const uint32_t tiles = (uint32_t)((m + TR - 1) / TR) * nct;
  const uint32_t G = gridDim.x, b = blockIdx.x;
  // XCD x takes the x-th eighth of the tiles (the first G % 8 one more): unaligned rows share lines with the next tile's
  const uint32_t x8 = b % 8, wid = x8 * (G / 8) + (x8 < G % 8 ? x8 : G % 8) + b / 8;
  const uint32_t part = wid / tiles, tile = wid - part * tiles, ct = tile % nct;
  const int64_t r0 = (int64_t)(tile / nct) * TR, c0 = (int64_t)ct * TC;
  const bool do_xn = ct == 0 && g.XN != nullptr;
  // this wave's segments; the last segment of the depth goes through guarded loads where it is not whole, or (rows
  // contiguous) where a lane's words may run past the last row: at every earlier depth those bytes are the next
  // depth's first rows (sak >= m), and the rows of E they feed are never stored
  const uint32_t nseg = (uint32_t)((k + 63) / 64), slot = part * NW + (uint32_t)w, slots = NW * (uint32_t)g.splits;
  const int seg0 = (int)((uint64_t)nseg * slot / slots), seg1 = (int)((uint64_t)nseg * (slot + 1) / slots);
  const bool guard_last = (k % 64) != 0 || (MODE == ROWS && (m % 4) != 0 && r0 + TR > m);
  const bool tail = guard_last && seg1 == (int)nseg && seg1 > seg0;
  const int nf = seg1 - seg0 - (tail ? 1 : 0);                              // segments read without guards

  const uint16_t* A = g.A;
  constexpr int NAP = MODE == ROWS ? 1 : TR / 8;
  const uint16_t* ap[NAP];
  if constexpr (MODE == ROWS) {
    const int64_t row = r0 + 4 * r;
    ap[0] = A + (row < m ? row : m - 4) + (64 * (int64_t)seg0 + 32 * h) * g.sak;
  } else {
#pragma unroll
    for (int I = 0; I < NAP; ++I) {
      const int64_t row = r0 + 8 * I + (lane >> 3);
      ap[I] = A + (row < m ? row : m - 1) * g.sam + 64 * (int64_t)seg0 + 8 * (lane & 7);
    }
  }
  const int64_t bstep = 3 * (int64_t)ncf * 512;
  const uint16_t* bq = (const uint16_t*)g.B + 4 * (int64_t)seg0 * bstep + 8 * lane;
  int bf[TCF];
#pragma unroll
  for (int n = 0; n < TCF; ++n) {
    const uint32_t f = (uint32_t)(c0 / 32) + n;
    bf[n] = (int)((f < ncf ? f : ncf - 1) * 512);
  }

  // ROWS: steps in flight, eight depths x 8 bytes; DEPTH: the next segment's 16 instructions
  uint32_t ra[MODE == ROWS ? 4 : 1][16];
  u32x4 as[MODE == ROWS ? 1 : NAP];
  u32x4 rb[4][3][TCF];
  auto load_a = [&](int j, int sg) {        // (ROWS) step j of this wave's segment sg
    const uint16_t* p = ap[0] + (64 * (int64_t)sg + 8 * j) * g.sak;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const u32x2 v = *reinterpret_cast<const u32x2_any*>(p + e * g.sak);
      ra[j][2 * e] = v.x;
      ra[j][2 * e + 1] = v.y;
    }
  };
  auto load_a_guarded = [&](int j, int sg) {                  // (ROWS) zeros past the depth and the rows
    const int64_t k0 = 64 * (int64_t)(seg0 + sg) + 32 * h + 8 * j;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      uint32_t v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int64_t row = r0 + 4 * r + i;
        v[i] = k0 + e < k && row < m ? A[(k0 + e) * g.sak + row] : 0u;
      }
      ra[j][2 * e] = v[0] | (v[1] << 16);
      ra[j][2 * e + 1] = v[2] | (v[3] << 16);
    }
  };
  uint8_t* const L = reinterpret_cast<uint8_t*>(red) + w * TR * 128;
  auto load_seg = [&](int sg) {             // (DEPTH) this wave's segment sg
#pragma unroll
    for (int I = 0; I < NAP; ++I) as[I] = *reinterpret_cast<const u32x4_lane*>(ap[I] + 64 * (int64_t)sg);
  };
  auto load_seg_guarded = [&](int sg) {     // (DEPTH) zeros past the depth
    const int64_t kk = 64 * (int64_t)(seg0 + sg) + 8 * (lane & 7);
#pragma unroll
    for (int I = 0; I < NAP; ++I) {
      const uint16_t* p = ap[I] + 64 * (int64_t)sg;
      if (k >= 8) {                         // the last 8 depths where these pass the end, those before kk dropped
        const int64_t over = kk + 8 - k > 0 ? kk + 8 - k : 0;
        as[I] = drop_low(*reinterpret_cast<const u32x4_lane*>(p - over), over < 8 ? (int)over : 8);
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          uint32_t v[2];
#pragma unroll
          for (int e = 0; e < 2; ++e) v[e] = kk + 2 * q + e < k ? p[2 * q + e] : 0u;
          as[I][q] = v[0] | (v[1] << 16);
        }
      }
    }
  };
  auto store_seg = [&]() {
    sdc_wave_lds_fence();
#pragma unroll
    for (int I = 0; I < NAP; ++I)
      *reinterpret_cast<u32x4*>(L + (8 * I + (lane >> 3)) * 128 + 16 * ((lane & 7) ^ (lane >> 3))) = as[I];
    sdc_wave_lds_fence();
  };
  auto load_b = [&](int j, int sg) {
    const uint16_t* p = bq + (4 * (int64_t)sg + j) * bstep;
#pragma unroll
    for (int q = 0; q < 3; ++q)
#pragma unroll
      for (int n = 0; n < TCF; ++n) rb[j][q][n] = *reinterpret_cast<const u32x4*>(p + (int64_t)q * ncf * 512 + bf[n]);
  };
  f32x16 acc[TRF][TCF];
  float xsq[TRF], xab[TRF];
#pragma unroll
  for (int i = 0; i < TRF; ++i) {
    xsq[i] = xab[i] = 0.f;
#pragma unroll
    for (int n = 0; n < TCF; ++n)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][n][e] = 0.f;
  }
  auto step = [&](int j) {
    u32x4 a[TRF];
    if constexpr (MODE == ROWS) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const uint32_t x0 = ra[j][4 * q], y0 = ra[j][4 * q + 1], x1 = ra[j][4 * q + 2], y1 = ra[j][4 * q + 3];
        a[0][q] = __builtin_amdgcn_perm(x1, x0, 0x05040100u);             // depths 2 q and 2 q + 1 of row 4 r
        a[1][q] = __builtin_amdgcn_perm(x1, x0, 0x07060302u);
        a[2][q] = __builtin_amdgcn_perm(y1, y0, 0x05040100u);
        a[3][q] = __builtin_amdgcn_perm(y1, y0, 0x07060302u);
      }
    } else {
#pragma unroll
      for (int i = 0; i < TRF; ++i)
        a[i] = *reinterpret_cast<const u32x4*>(L + (32 * i + r) * 128 + 16 * ((4 * h + j) ^ (r & 7)));
    }
#pragma unroll
    for (int p = 0; p < 3; ++p)
#pragma unroll
      for (int n = 0; n < TCF; ++n)
#pragma unroll
        for (int i = 0; i < TRF; ++i) acc[i][n] = sdc_pipe::mfma32<DT>(a[i], rb[j][p][n], acc[i][n]);
    if (do_xn) {
      constexpr uint32_t ONES = DT == SDC_BF16 ? 0x3F803F80u : 0x3C003C00u;
#pragma unroll
      for (int i = 0; i < TRF; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          xsq[i] = pk_dot2<DT>(a[i][q], a[i][q], xsq[i]);
          xab[i] = pk_dot2<DT>(a[i][q] & 0x7FFF7FFFu, ONES, xab[i]);
        }
    }
  };
  if constexpr (MODE == ROWS) {
    if (nf > 0) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        load_a(j, 0);
        load_b(j, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
      for (int sg = 0; sg < nf; ++sg) {
        const int nx = sg + 1 < nf ? sg + 1 : nf - 1;                      // (past the last: the last again)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          step(j);
          __builtin_amdgcn_sched_barrier(0);
          load_a(j, nx);
          load_b(j, nx);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    if (tail) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        load_a_guarded(j, nf);
        load_b(j, nf);
        step(j);
      }
    }
  } else if (seg1 > seg0) {
    // (the wave's LDS holds one segment, stored by some lanes and read by others)
    if (nf > 0) {
      load_seg(0);
#pragma unroll
      for (int j = 0; j < 4; ++j) load_b(j, 0);
      store_seg();
      for (int sg = 0; sg < nf; ++sg) {
        const int nx = sg + 1 < nf ? sg + 1 : nf - 1;                      // (past the last: the last again)
        load_seg(nx);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          step(j);
          __builtin_amdgcn_sched_barrier(0);
          load_b(j, nx);
          __builtin_amdgcn_sched_barrier(0);
        }
        store_seg();
      }
    }
    if (tail) {
      load_seg_guarded(nf);
#pragma unroll
      for (int j = 0; j < 4; ++j) load_b(j, nf);
      store_seg();
#pragma unroll
      for (int j = 0; j < 4; ++j) step(j);
    }
  }
  if constexpr (MODE == DEPTH) __syncthreads();       // (the epilogue's LDS overlaps other waves' segments)
  // fragment row x of fragment i is row 4 x + i of the tile (rows contiguous), or 32 i + x
  if (do_xn) {
#pragma unroll
    for (int i = 0; i < TRF; ++i) {
      xsq[i] += __shfl_xor(xsq[i], 32, 64);
      xab[i] += __shfl_xor(xab[i], 32, 64);
      if (h == 0) {
        const int row = MODE == ROWS ? 4 * r + i : 32 * i + r;
        xred[w][row][0] = xsq[i];
        xred[w][row][1] = xab[i];
      }
    }
  }
  // the waves' sums in LDS, [wave][column][row] (rows padded to RP), then added in wave order
#pragma unroll
  for (int n = 0; n < TCF; ++n)
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) {
      float* col = red + (w * TC + 32 * n + r) * RP;
      if constexpr (MODE == ROWS) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          *reinterpret_cast<f32x4*>(col + 4 * (8 * r4 + 4 * h + e)) =
              f32x4{acc[0][n][4 * r4 + e], acc[1][n][4 * r4 + e], acc[2][n][4 * r4 + e], acc[3][n][4 * r4 + e]};
      } else {
#pragma unroll
        for (int i = 0; i < TRF; ++i)
          *reinterpret_cast<f32x4*>(col + 32 * i + 8 * r4 + 4 * h) =
              f32x4{acc[i][n][4 * r4], acc[i][n][4 * r4 + 1], acc[i][n][4 * r4 + 2], acc[i][n][4 * r4 + 3]};
      }
    }
  __syncthreads();
  if (do_xn && t < TR && r0 + t < m) {
    float sq = xred[0][t][0], ab = xred[0][t][1];
#pragma unroll
    for (int q = 1; q < NW; ++q) {
      sq += xred[q][t][0];
      ab += xred[q][t][1];
    }
    g.XN[part * 2 * m + r0 + t] = sq;
    g.XN[part * 2 * m + m + r0 + t] = ab;
  }
  float* const Ep = g.E + part * N * m;
  if (g.et) {
    // transposed plane [N][m]: an instruction writes two whole columns of the tile, lane l rows 4 (l % 32) .. + 3
#pragma unroll
    for (int gq = 0; gq < TC / (2 * NW); ++gq) {
      const int cl = (w * (TC / (2 * NW)) + gq) * 2 + (lane >> 5);
      f32x4 v = *reinterpret_cast<const f32x4*>(red + cl * RP + 4 * (lane & 31));
#pragma unroll
      for (int q = 1; q < NW; ++q) v += *reinterpret_cast<const f32x4*>(red + (q * TC + cl) * RP + 4 * (lane & 31));
      const int64_t row = r0 + 4 * (lane & 31), col = c0 + cl;
      if (col < N) {
        float* Ec = Ep + col * m;
        if (row + 4 <= m && m % 4 == 0) {
          *reinterpret_cast<f32x4*>(Ec + row) = v;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (row + e < m) Ec[row + e] = v[e];
        }
      }
    }
  } else {
    // row-major plane [m][N]: an instruction writes whole rows of the tile, lane l four columns of one (RowMajor)
    using Map = RowMajor<TCF>;
    const int c4 = Map::col(lane);
#pragma unroll
    for (int gq = 0; gq < Map::STEPS; ++gq) {
      const int rl = Map::row(w, gq, lane);
      f32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float x = red[(c4 + e) * RP + rl];
#pragma unroll
        for (int q = 1; q < NW; ++q) x += red[(q * TC + c4 + e) * RP + rl];
        v[e] = x;
      }
      const int64_t row = r0 + rl, col = c0 + c4;
      if (row < m) {
        float* Er = Ep + row * N;
        if (col + 4 <= N && N % 4 == 0) {
          *reinterpret_cast<f32x4*>(Er + col) = v;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (col + e < N) Er[col + e] = v[e];
        }
      }
    }
  }
  if (blockIdx.x == 0) sdc_clear_slots(g.slots, g.slot_sets, t, 64 * NW);
}

template <int DT, int TCF>
void lane_launch_mode(bool rows, dim3 grid, const GemmArgs& g, hipStream_t stream) {
  const dim3 block(64 * NW);
  if (rows) hipLaunchKernelGGL((lane_gemm_kernel<DT, ROWS, TCF>), grid, block, 0, stream, g);
  else hipLaunchKernelGGL((lane_gemm_kernel<DT, DEPTH, TCF>), grid, block, 0, stream, g);
}

template <int DT>
void lane_launch(bool rows, int tcf, dim3 grid, const GemmArgs& g, hipStream_t stream) {
  if (tcf == 1) lane_launch_mode<DT, 1>(rows, grid, g, stream);
  else lane_launch_mode<DT, 2>(rows, grid, g, stream);
}

}  // namespace

// Columns of this GEMM's tiles: an output of at most 32 would leave half of a wider tile's products empty
static int sdc_lane_gemm_columns(int64_t N) { return N <= 32 ? 32 : 64; }

// E (and, with g.XN, A's row norms) for one batch of a 16-bit A with unit depth stride, or unit row stride and
// disjoint depths (g.sak >= g.m >= 4); B in fragment order for the depth rounded up to 64, zeros past it; g.splits
// (1 .. SDC_MAX_GEMM_SPLITS) planes.  Returns SDC_EUNSUPPORTED, launching nothing, for other strides.
int sdc_lane_gemm_launch(int dtype, GemmArgs g, hipStream_t stream) {
  if (dtype != SDC_BF16 && dtype != SDC_FP16) return SDC_EUNSUPPORTED;
  const bool rows = g.sak != 1 && g.sam == 1 && g.sak >= g.m && g.m >= 4;
  if (g.sak != 1 && !rows) return SDC_EUNSUPPORTED;
  if (g.goffs || g.xf_blocks || g.splits < 1 || g.splits > SDC_MAX_GEMM_SPLITS || (uintptr_t)g.B % 16 ||
      (uintptr_t)g.A % 2 || (uintptr_t)g.E % 16 || g.k < 1 || g.k > (1ll << 31))
    return SDC_EUNSUPPORTED;
  if (g.m < 1 || g.N < 1) return SDC_EINVAL;
  const int tcf = sdc_lane_gemm_columns(g.N) / 32;
  const int64_t blocks = g.splits * sdc_cdiv(g.m, TR) * sdc_cdiv(g.N, 32 * tcf);
  if (blocks > 0x7FFFFFFF || g.N > 0x7FFFFFFF) return SDC_EUNSUPPORTED;
  SdcProf prof(g.prof_name ? g.prof_name : "expected_gemm", stream);
  const dim3 grid((unsigned)blocks);
  if (dtype == SDC_BF16) lane_launch<SDC_BF16>(rows, tcf, grid, g, stream);
  else lane_launch<SDC_FP16>(rows, tcf, grid, g, stream);
  SDC_LAUNCH_CHECK();
  return SDC_OK;
}
