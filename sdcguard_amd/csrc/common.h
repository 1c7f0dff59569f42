// Shared device helpers for the sdcguard HIP kernels (gfx950, wave64).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define SDC_WAVE 64
// most depth-split planes of the expected-side GEMM (its scorers add them with unrolled loads)
#define SDC_MAX_SPLITS 8
// depth splits the expected-side GEMMs accept (a scoring pass holds SDC_MAX_SPLITS splits' values in registers and
// loops over those past them: short GEMMs, whose planes are small)
#define SDC_MAX_GEMM_SPLITS 32

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef int32_t i32x4 __attribute__((ext_vector_type(4)));
typedef int32_t i32x16 __attribute__((ext_vector_type(16)));

// Element kinds of the checked matmul's operands.  The expected-side GEMM also runs in two quantized modes:
// SDC_FP8 (A fp8 e4m3, converted exactly to bf16 on load; bf16 parts) and SDC_I8 (A int8; int8 parts).
enum SdcDtype { SDC_BF16 = 0, SDC_FP16 = 1, SDC_FP8 = 2, SDC_I8 = 3 };

// Status codes of the C ABI.
enum SdcStatus {
  SDC_OK = 0,
  SDC_EINVAL = -1,        // an argument is out of range (shape, stride, null pointer)
  SDC_EUNSUPPORTED = -2,  // a case this library does not implement (the caller must not pretend it ran)
  SDC_EWORKSPACE = -3,    // the workspace is smaller than the matching *_workspace() call asked for
  SDC_ELAUNCH = -4,       // a HIP launch error
};

__device__ __forceinline__ float bf16_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) { return __uint_as_float(w & 0xFFFF0000u); }
__device__ __forceinline__ float f16_lo(uint32_t w) {
  _Float16 h = __builtin_bit_cast(_Float16, (uint16_t)(w & 0xFFFFu));
  return (float)h;
}
__device__ __forceinline__ float f16_hi(uint32_t w) {
  _Float16 h = __builtin_bit_cast(_Float16, (uint16_t)(w >> 16));
  return (float)h;
}

template <int DT>
__device__ __forceinline__ float lo_of(uint32_t w) { return DT == SDC_BF16 ? bf16_lo(w) : f16_lo(w); }
template <int DT>
__device__ __forceinline__ float hi_of(uint32_t w) { return DT == SDC_BF16 ? bf16_hi(w) : f16_hi(w); }
template <int DT>
__device__ __forceinline__ float half_to_f32(uint16_t h) {
  return DT == SDC_BF16 ? __uint_as_float((uint32_t)h << 16) : (float)__builtin_bit_cast(_Float16, h);
}

// DPP lane exchange inside a quad (xor 1 / xor 2): one VALU op each, no LDS traffic.
__device__ __forceinline__ float dpp_xor1(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, false));
}
__device__ __forceinline__ float dpp_xor2(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xF, 0xF, false));
}
__device__ __forceinline__ float quad_sum(float v) {
  v += dpp_xor1(v);
  v += dpp_xor2(v);
  return v;
}

__device__ __forceinline__ int64_t shfl_xor_i64(int64_t v, int mask) {
  int lo = (int)(uint32_t)(uint64_t)v;
  int hi = (int)(uint32_t)((uint64_t)v >> 32);
  lo = __shfl_xor(lo, mask, SDC_WAVE);
  hi = __shfl_xor(hi, mask, SDC_WAVE);
  return (int64_t)(((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo);
}

__device__ __forceinline__ int64_t wave_max_i64(int64_t v) {
#pragma unroll
  for (int m = 1; m < SDC_WAVE; m <<= 1) {
    int64_t o = shfl_xor_i64(v, m);
    v = o > v ? o : v;
  }
  return v;
}

__device__ __forceinline__ int64_t wave_sum_i64(int64_t v) {
#pragma unroll
  for (int m = 1; m < SDC_WAVE; m <<= 1) v += shfl_xor_i64(v, m);
  return v;
}

__device__ __forceinline__ int wave_sum_i32(int v) {
#pragma unroll
  for (int m = 1; m < SDC_WAVE; m <<= 1) v += __shfl_xor(v, m, SDC_WAVE);
  return v;
}

__device__ __forceinline__ float wave_sum_f32(float v) {
#pragma unroll
  for (int m = 1; m < SDC_WAVE; m <<= 1) v += __shfl_xor(v, m, SDC_WAVE);
  return v;
}

// Wave reductions on DPP lane moves: xor 1 and xor 2 (quad swaps), the half-row and row mirrors (every lane of a
// row of 16 then holds its row's result), then the four rows read through lanes 0, 16, 32 and 48.  No LDS round
// trips, unlike the shuffles above; every lane of the wave must be active.  (Integer maxima and sums: any order
// gives the same result.)
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, false);
}
__device__ __forceinline__ uint32_t wave_max_u32_dpp(uint32_t v) {
  v = max(v, dpp_u32<0xB1>(v));
  v = max(v, dpp_u32<0x4E>(v));
  v = max(v, dpp_u32<0x141>(v));
  v = max(v, dpp_u32<0x140>(v));
  const uint32_t a = (uint32_t)__builtin_amdgcn_readlane((int)v, 0), b = (uint32_t)__builtin_amdgcn_readlane((int)v, 16);
  const uint32_t c = (uint32_t)__builtin_amdgcn_readlane((int)v, 32), d = (uint32_t)__builtin_amdgcn_readlane((int)v, 48);
  return max(max(a, b), max(c, d));
}
__device__ __forceinline__ int wave_sum_i32_dpp(int v) {
  v += (int)dpp_u32<0xB1>((uint32_t)v);
  v += (int)dpp_u32<0x4E>((uint32_t)v);
  v += (int)dpp_u32<0x141>((uint32_t)v);
  v += (int)dpp_u32<0x140>((uint32_t)v);
  return (__builtin_amdgcn_readlane(v, 0) + __builtin_amdgcn_readlane(v, 16)) +
         (__builtin_amdgcn_readlane(v, 32) + __builtin_amdgcn_readlane(v, 48));
}
// (Float sums: the order is the lanes' pairs, then quads, eights and rows, then the rows in pairs.)
__device__ __forceinline__ float wave_sum_f32_dpp(float v) {
  v += __uint_as_float(dpp_u32<0xB1>(__float_as_uint(v)));
  v += __uint_as_float(dpp_u32<0x4E>(__float_as_uint(v)));
  v += __uint_as_float(dpp_u32<0x141>(__float_as_uint(v)));
  v += __uint_as_float(dpp_u32<0x140>(__float_as_uint(v)));
  const float a = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 0));
  const float b = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 16));
  const float c = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 32));
  const float d = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 48));
  return (a + b) + (c + d);
}
__device__ __forceinline__ float wave_max_f32_dpp(float v) {
  v = fmaxf(v, __uint_as_float(dpp_u32<0xB1>(__float_as_uint(v))));
  v = fmaxf(v, __uint_as_float(dpp_u32<0x4E>(__float_as_uint(v))));
  v = fmaxf(v, __uint_as_float(dpp_u32<0x141>(__float_as_uint(v))));
  v = fmaxf(v, __uint_as_float(dpp_u32<0x140>(__float_as_uint(v))));
  const float a = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 0));
  const float b = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 16));
  const float c = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 32));
  const float d = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 48));
  return fmaxf(fmaxf(a, b), fmaxf(c, d));
}
template <int CTRL>
__device__ __forceinline__ int64_t dpp_i64(int64_t v) {
  const uint32_t lo = dpp_u32<CTRL>((uint32_t)(uint64_t)v), hi = dpp_u32<CTRL>((uint32_t)((uint64_t)v >> 32));
  return (int64_t)(((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ int64_t readlane_i64(int64_t v, int l) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(uint64_t)v, l);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)((uint64_t)v >> 32), l);
  return (int64_t)(((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ int64_t wave_max_i64_dpp(int64_t v) {
  int64_t o = dpp_i64<0xB1>(v);
  v = o > v ? o : v;
  o = dpp_i64<0x4E>(v);
  v = o > v ? o : v;
  o = dpp_i64<0x141>(v);
  v = o > v ? o : v;
  o = dpp_i64<0x140>(v);
  v = o > v ? o : v;
  int64_t r = readlane_i64(v, 0);
#pragma unroll
  for (int l = 16; l < 64; l += 16) {
    const int64_t q = readlane_i64(v, l);
    r = q > r ? q : r;
  }
  return r;
}

// Between a wave's LDS stores and another lane's loads of them (and between loads and the stores that follow), where the wave
// is the only one at that memory.  A wave's LDS accesses are done in order, so no instruction comes of it, but without it
// the compiler, which orders one lane's accesses only, may move them past each other.
__device__ __forceinline__ void sdc_wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// The worst keys of a check's result row (res[0]: key, res[1]: key with its noise; both hold the score's bits in
// their high half), raised by one thread of a workgroup.  Device-scope maxima on one address from every XCD
// serialize at about 14 ns each: on a row that starts at zero, as every queued check's does, two for each of a
// pass's thousands of workgroups took longer than the pass (fp8 4096 x 14336: 227 us; the linear check's pass over
// y: 100 us).  So a workgroup first raises a slot that only its own XCD uses (the line stays in that XCD's L2; the
// slots are cleared by a kernel earlier in the call: sdc_clear_slots), and goes on to the row only with a key that
// was the slot's largest so far, about ln(workgroups / 8) times a slot: 41 us and 35 us (32 slots picked by the
// workgroup's number: 73 and 54 us).  The largest key of all is the largest of its slot whenever it comes, so it
// always reaches the row, whichever slots the workgroups took.  A lower score than the slot's cannot raise either
// word.  seen0, seen1: the row's keys read earlier (keys only grow: a stale value only lets a maximum through).
constexpr int SDC_SLOTS = 8;                                             // one per XCD
constexpr int SDC_SLOT_WORDS = 16;                                       // 128 bytes each
constexpr int SDC_SLOT_FLOATS = SDC_SLOTS * SDC_SLOT_WORDS * 2;          // workspace of a set of slots, in floats
__device__ __forceinline__ void sdc_raise_worst(int64_t* res, unsigned long long* slots, int64_t key, int64_t keyd,
                                                int64_t seen0, int64_t seen1) {
  if (key <= seen0 && keyd <= seen1) return;
  if (!slots) {                                                          // (a pass of few workgroups)
    if (key > seen0) atomicMax((unsigned long long*)res, (unsigned long long)key);
    if (keyd > seen1) atomicMax((unsigned long long*)(res + 1), (unsigned long long)keyd);
    return;
  }
  const uint32_t xcc = __builtin_amdgcn_s_getreg(20 | (3 << 11));        // HW_REG_XCC_ID, bits 0 .. 3
  unsigned long long* s = slots + SDC_SLOT_WORDS * (xcc % SDC_SLOTS);
  const unsigned long long k0 = (unsigned long long)key, k1 = (unsigned long long)keyd;
  const unsigned long long o0 = atomicMax(s, k0);
  if ((k0 >> 32) < (o0 >> 32)) return;
  const unsigned long long o1 = atomicMax(s + 1, k1);
  if (k0 > o0 && key > seen0) atomicMax((unsigned long long*)res, k0);
  if (k1 > o1 && keyd > seen1) atomicMax((unsigned long long*)(res + 1), k1);
}
// The slots for a pass of `raisers` workgroups (or waves, where each raises the row itself), none for a few: a slot's
// maxima have to return before the workgroup ends, the row's own are sent off unwaited.  Measured into fresh rows, with
// slots and without, by workgroups: y pass 16 5.5 and 4.8 us, 48 5.5 and 5.3, 64 5.5 and 5.6, 256 5.5 and 10.0; training
// scores 16 6.4 and 5.8, 48 7.4 and 6.9, 64 7.3 and 7.6, 256 8.4 and 11.2; precise scores 32 10.0 and 9.7, 64 9.9 and
// 10.1, 256 10.2 and 14.7; fp8 tiles (two waves a workgroup) 16 5.9 and 5.6, 30 5.9 and 6.1, 64 6.0 and 7.8.
constexpr int64_t SDC_SLOT_RAISERS = 64;
static inline unsigned long long* sdc_slots_for(int64_t raisers, unsigned long long* slots) {
  return raisers < SDC_SLOT_RAISERS ? nullptr : slots;
}
// (called by every thread of one workgroup of an earlier kernel, at its end: nothing there waits for the stores; at its
// start they kept the one workgroup a microsecond behind the others, of 28 us for a whole 1024^3 check; `sets` sets
// of slots, null: none)
__device__ __forceinline__ void sdc_clear_slots(unsigned long long* slots, int sets, int t, int threads) {
  if (slots)
    for (int i = t; i < sets * SDC_SLOTS * SDC_SLOT_WORDS; i += threads) slots[i] = 0ull;
}

// bits of a float as an int64 holding the unsigned 32-bit pattern
__device__ __forceinline__ int64_t fbits64(float f) { return (int64_t)(uint32_t)__float_as_uint(f); }

__host__ __device__ static inline int64_t sdc_cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

// The HIP error behind the last SDC_ELAUNCH of this thread (sdc_last_error()).
void sdc_note_error(hipError_t e);

#define SDC_LAUNCH_CHECK()                                      \
  do {                                                          \
    hipError_t e_ = hipGetLastError();                          \
    if (e_ != hipSuccess) {                                     \
      sdc_note_error(e_);                                       \
      return SDC_ELAUNCH;                                       \
    }                                                           \
  } while (0)

// Entry points clear errors left by earlier HIP calls of the thread, so a launch check sees only its own.
#define SDC_CLEAR_ERRORS() (void)hipGetLastError()
