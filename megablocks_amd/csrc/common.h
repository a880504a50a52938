// Shared helpers for the libmbx kernels (gfx950, wave64).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "../../include/mbx.h"

namespace mbx {

constexpr int kWave = 64;

#define MBX_HIP_CHECK(expr)                  \
  do {                                       \
    hipError_t e_ = (expr);                  \
    if (e_ != hipSuccess) return (int)e_;    \
  } while (0)

// Returns the launch status of the kernel(s) just enqueued.
static inline int launch_status() { return (int)hipGetLastError(); }

static inline hipStream_t as_stream(mbx_stream_t s) { return (hipStream_t)s; }

static inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// ---- storage <-> fp32 conversions (round-to-nearest-even, like torch) ----
typedef uint16_t bf16_t;  // raw bits
typedef _Float16 f16_t;

__device__ __forceinline__ float bf16_to_f32(uint16_t v) { return __uint_as_float(((uint32_t)v) << 16); }

__device__ __forceinline__ uint16_t f32_to_bf16(float f) {
  return __builtin_bit_cast(uint16_t, (__bf16)f);   // v_cvt_pk_bf16_f32: round to nearest even, NaN stays NaN
}

template <int DT> struct Elem;
template <> struct Elem<MBX_BF16> {
  typedef uint16_t type;
  static __device__ __forceinline__ float to_f32(type v) { return bf16_to_f32(v); }
  static __device__ __forceinline__ type from_f32(float f) { return f32_to_bf16(f); }
};
template <> struct Elem<MBX_F16> {
  typedef _Float16 type;
  static __device__ __forceinline__ float to_f32(type v) { return (float)v; }
  static __device__ __forceinline__ type from_f32(float f) { return (_Float16)f; }
};
template <> struct Elem<MBX_F32> {
  typedef float type;
  static __device__ __forceinline__ float to_f32(type v) { return v; }
  static __device__ __forceinline__ type from_f32(float f) { return f; }
};

static inline int dtype_bytes(int dtype) { return dtype == MBX_F32 ? 4 : 2; }
static inline int itype_bytes(int itype) { return itype == MBX_I16 ? 2 : (itype == MBX_I32 ? 4 : 8); }

// Reads element i of an array of runtime dtype as fp32 (used for the per-row router weight).
__device__ __forceinline__ float load_as_f32(const void* p, int64_t i, int dtype) {
  if (dtype == MBX_BF16) return bf16_to_f32(((const uint16_t*)p)[i]);
  if (dtype == MBX_F16) return (float)((const _Float16*)p)[i];
  return ((const float*)p)[i];
}

// ---- wave64 primitives ----
__device__ __forceinline__ int lane_id() { return __lane_id(); }

// Between lanes without the LDS: a shuffle (ds_bpermute_b32) keeps a wave waiting some 100 cycles, a permute or DPP
// operand two or three instructions, and a reduction is six of them in a chain.
//
// wave_butterfly(v, op): all lanes get v combined over the wave, op(v, v of the lane 32, 16, 8, 4, 2, 1 further) in turn, for a
// commutative op.  The steps by 32 and 16 swap half waves and rows of 16; by 8 the row is rotated by 8, by 4 by 4 (its
// halves are alike by then), by 2 and 1 quads are permuted.  All lanes must be active.
template <int STEP>
__device__ __forceinline__ uint32_t lane_xor_dpp(uint32_t v) {   // STEP 8 (4: lanes 8 apart are alike), 2, 1
  constexpr int ctrl = STEP == 8 ? 0x128 : STEP == 4 ? 0x124 : STEP == 2 ? 0x4e : 0xb1;
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, ctrl, 0xf, 0xf, true);
}
template <typename T, typename F>
__device__ __forceinline__ T wave_butterfly(T v, F&& op) {
  static_assert(sizeof(T) == 4, "one register");
  const auto bits = [](T x) { return __builtin_bit_cast(uint32_t, x); };
  const auto value = [](uint32_t x) { return __builtin_bit_cast(T, x); };
  const auto halves = __builtin_amdgcn_permlane32_swap(bits(v), bits(v), false, false);
  v = op(value(halves[0]), value(halves[1]));
  const auto rows = __builtin_amdgcn_permlane16_swap(bits(v), bits(v), false, false);
  v = op(value(rows[0]), value(rows[1]));
  v = op(v, value(lane_xor_dpp<8>(bits(v))));
  v = op(v, value(lane_xor_dpp<4>(bits(v))));
  v = op(v, value(lane_xor_dpp<2>(bits(v))));
  return op(v, value(lane_xor_dpp<1>(bits(v))));
}

__device__ __forceinline__ float wave_sum(float v) {
  return wave_butterfly(v, [](float a, float b) { return a + b; });
}
__device__ __forceinline__ float wave_max(float v) {
  return wave_butterfly(v, [](float a, float b) { return fmaxf(a, b); });
}
__device__ __forceinline__ int wave_max(int v) {
  return wave_butterfly(v, [](int a, int b) { return a > b ? a : b; });
}

// Lane `from`'s value, the same `from` in all lanes.
__device__ __forceinline__ int lane_value(int v, int from) { return __builtin_amdgcn_readlane(v, from); }
__device__ __forceinline__ float lane_value(float v, int from) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), from)); }

// Inclusive prefix sum across the 64 lanes of a wave.
template <typename T>
__device__ __forceinline__ T wave_inclusive_scan(T v) {
  if constexpr (sizeof(T) == 4) {
    const auto moved = [](T x, auto ctrl, auto rows) {   // zero where no lane is that far below, in the rows not named
      return (T)__builtin_amdgcn_update_dpp(0, (int)x, decltype(ctrl)::value, decltype(rows)::value, 0xf, false);
    };
    typedef std::integral_constant<int, 0xf> all;
    v += moved(v, std::integral_constant<int, 0x111>{}, all{});   // row_shr by 1, 2, 4, 8: inside the rows of 16
    v += moved(v, std::integral_constant<int, 0x112>{}, all{});
    v += moved(v, std::integral_constant<int, 0x114>{}, all{});
    v += moved(v, std::integral_constant<int, 0x118>{}, all{});
    v += moved(v, std::integral_constant<int, 0x142>{}, std::integral_constant<int, 0xa>{});   // row_bcast:15 to rows 1 and 3
    v += moved(v, std::integral_constant<int, 0x143>{}, std::integral_constant<int, 0xc>{});   // row_bcast:31 to rows 2 and 3
  } else {
    const int lane = lane_id();
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      T o = __shfl_up(v, off, 64);
      if (lane >= off) v += o;
    }
  }
  return v;
}

// First e in [0, n) with bins[e] > r (bins inclusive cumsum, non-decreasing); n if none.
__device__ __forceinline__ int upper_bound_i32(const int32_t* __restrict__ bins, int n, int r) {
  int lo = 0, hi = n;
  while (lo < hi) {
    int mid = (lo + hi) >> 1;
    if (bins[mid] > r) hi = mid; else lo = mid + 1;
  }
  return lo;
}

}  // namespace mbx
