// Shared device-side helpers for the gfx950 kernels: vector types, fp8 / bf16
// conversions built on the CDNA4 conversion instructions, wave reductions.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/mi355q.h"

namespace mi355q {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

constexpr float kFp8Max[2] = {448.0f, 57344.0f};  // e4m3fn, e5m2

// Dynamic per-row quantisation computes scale = target / amax.  A row of zeros
// (amax 0) or of values so small that the quotient overflows would give an
// infinite scale, and 0 * inf = NaN would turn every zero of the row into an
// fp8 NaN.  The scale is therefore capped at the largest finite bf16 value
// (0x7f7f0000; finite in fp32 and after the rounding to bf16 that a bf16 input
// applies to it): a zero row then gives zero codes and a finite 1 / scale.  A
// NaN amax (a NaN in the row) compares false and stays NaN.
constexpr float kRowScaleCap = 3.3895313892515355e38f;
__device__ __forceinline__ float row_scale(float target, float amax) {
  const float s = target / amax;  // correctly rounded fp32 division, as on the host
  return s > kRowScaleCap ? kRowScaleCap : s;
}

__device__ __forceinline__ float bf16_bits_to_f32(uint32_t h) { return __uint_as_float(h << 16); }

// fp32 -> bf16 round-to-nearest-even (v_cvt_pk_bf16_f32), returned as fp32.
__device__ __forceinline__ float round_to_bf16(float v) {
  __bf16 h = (__bf16)v;
  return (float)h;
}

// two fp32 -> packed bf16 pair (lo = a, hi = b)
__device__ __forceinline__ uint32_t pack_bf16x2(float a, float b) {
  bf16x2 r = {(__bf16)a, (__bf16)b};
  return __builtin_bit_cast(uint32_t, r);
}

// x / (1 + exp(-x)) for a bf16 x, accurate enough that rounding the result to bf16 gives the bits of the CPU
// oracle's fixed sequence of IEEE operations for every one of the 65536 values x can take (a test compares them all).
// With t = |x| exp(-|x|) / (1 + exp(-|x|)) it is max(x, -0) - t: nothing overflows and nothing cancels.  The
// exponential carries a factor of 2, which keeps it a normal number down to x = -88, the last value with a result;
// below that v_exp_f32 gives 0 and the result is -0.  -inf gives inf * 0 = NaN, and a NaN passes through the maximum.
// Nine instructions, two of them transcendental; the IEEE sequence took fifty.
__device__ __forceinline__ float silu_for_bf16(float x) {
  const float xm = __builtin_fminf(x, 128.0f);
  const float e = __builtin_amdgcn_exp2f(__builtin_fmaf(__builtin_fabsf(xm), -1.44269504088896341f, 1.0f));
  const float p = __builtin_fabsf(xm) * (e * __builtin_amdgcn_rcpf(__builtin_fmaf(e, 0.5f, 1.0f)));
  return __builtin_fmaf(-p, 0.5f, __builtin_elementwise_maximum(x, -0.0f));
}

// Clamp to the finite fp8 range.  minimum/maximum propagate NaN, so a NaN
// input still converts to an fp8 NaN; +-Inf saturates like any overflow.
template <int FMT>
__device__ __forceinline__ float sat_fp8(float v) {
  constexpr float mx = (FMT == MI355Q_E5M2) ? 57344.0f : 448.0f;
  return __builtin_elementwise_minimum(__builtin_elementwise_maximum(v, -mx), mx);
}

// four fp32 -> four fp8 bytes (element 0 in the low byte), RNE, saturating.
// The raw v_cvt_pk_{fp8,bf8}_f32 turns overflow into NaN/Inf, hence the clamp.
template <int FMT>
__device__ __forceinline__ uint32_t cvt_fp8x4(float a, float b, float c, float d) {
  a = sat_fp8<FMT>(a);
  b = sat_fp8<FMT>(b);
  c = sat_fp8<FMT>(c);
  d = sat_fp8<FMT>(d);
  int r;
  if constexpr (FMT == MI355Q_E5M2) {
    r = __builtin_amdgcn_cvt_pk_bf8_f32(a, b, 0, false);
    r = __builtin_amdgcn_cvt_pk_bf8_f32(c, d, r, true);
  } else {
    r = __builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false);
    r = __builtin_amdgcn_cvt_pk_fp8_f32(c, d, r, true);
  }
  return (uint32_t)r;
}

// The same for values known to lie below the halfway point past the largest finite code (464; 61440), which round to
// that code by themselves: what a row scaled by target / amax with |target| <= the largest finite value holds, whatever
// the roundings on the way (at most 450; 57600).  NaN stays NaN.
template <int FMT>
__device__ __forceinline__ uint32_t cvt_fp8x4_in_range(float a, float b, float c, float d) {
  int r;
  if constexpr (FMT == MI355Q_E5M2) {
    r = __builtin_amdgcn_cvt_pk_bf8_f32(a, b, 0, false);
    r = __builtin_amdgcn_cvt_pk_bf8_f32(c, d, r, true);
  } else {
    r = __builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false);
    r = __builtin_amdgcn_cvt_pk_fp8_f32(c, d, r, true);
  }
  return (uint32_t)r;
}

// Stochastic rounding of four fp32 to fp8 (v_cvt_sr_fp8_f32 / v_cvt_sr_bf8_f32:
// the 32 random bits are added below the kept mantissa before truncation), after
// the same saturating clamp as the round-to-nearest path.
template <int FMT>
__device__ __forceinline__ uint32_t cvt_fp8x4_sr(float a, float b, float c, float d, uint32_t r0,
                                                 uint32_t r1, uint32_t r2, uint32_t r3) {
  a = sat_fp8<FMT>(a);
  b = sat_fp8<FMT>(b);
  c = sat_fp8<FMT>(c);
  d = sat_fp8<FMT>(d);
  int r = 0;
  if constexpr (FMT == MI355Q_E5M2) {
    r = __builtin_amdgcn_cvt_sr_bf8_f32(a, r0, r, 0);
    r = __builtin_amdgcn_cvt_sr_bf8_f32(b, r1, r, 1);
    r = __builtin_amdgcn_cvt_sr_bf8_f32(c, r2, r, 2);
    r = __builtin_amdgcn_cvt_sr_bf8_f32(d, r3, r, 3);
  } else {
    r = __builtin_amdgcn_cvt_sr_fp8_f32(a, r0, r, 0);
    r = __builtin_amdgcn_cvt_sr_fp8_f32(b, r1, r, 1);
    r = __builtin_amdgcn_cvt_sr_fp8_f32(c, r2, r, 2);
    r = __builtin_amdgcn_cvt_sr_fp8_f32(d, r3, r, 3);
  }
  return (uint32_t)r;
}

// 64 random bits for counter `idx` of stream `seed` (the splitmix64 finaliser:
// stateless, so an element's bits depend only on its index and the seed).
__device__ __forceinline__ uint64_t counter_random64(uint64_t seed, uint64_t idx) {
  uint64_t z = seed + (idx + 1) * 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

// four fp8 bytes of one dword -> four fp32 (exact)
template <int FMT>
__device__ __forceinline__ void cvt_f32x4(uint32_t w, float& a, float& b, float& c, float& d) {
  f32x2 lo, hi;
  if constexpr (FMT == MI355Q_E5M2) {
    lo = __builtin_amdgcn_cvt_pk_f32_bf8((int)w, false);
    hi = __builtin_amdgcn_cvt_pk_f32_bf8((int)w, true);
  } else {
    lo = __builtin_amdgcn_cvt_pk_f32_fp8((int)w, false);
    hi = __builtin_amdgcn_cvt_pk_f32_fp8((int)w, true);
  }
  a = lo.x; b = lo.y; c = hi.x; d = hi.y;
}

template <int FMT>
__device__ __forceinline__ float cvt_f32x1(uint32_t byte) {
  if constexpr (FMT == MI355Q_E5M2) return __builtin_amdgcn_cvt_f32_bf8((int)byte, 0);
  else return __builtin_amdgcn_cvt_f32_fp8((int)byte, 0);
}

// The largest of 16 neighbouring lanes' values, in each of them: lane i against i ^ 1, i ^ 2, then 7 - i and 15 - i, whose quads
// and eights are equal in themselves by then.
template <int DPP>
__device__ __forceinline__ uint32_t max_with_lane(uint32_t v) {
  const uint32_t o = (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, DPP, 0xf, 0xf, false);
  return v > o ? v : o;
}
__device__ __forceinline__ uint32_t row_max_u32(uint32_t v) {
  v = max_with_lane<0xb1>(v);     // quad_perm 1 0 3 2
  v = max_with_lane<0x4e>(v);     // quad_perm 2 3 0 1
  v = max_with_lane<0x141>(v);    // row_half_mirror
  return max_with_lane<0x140>(v);  // row_mirror
}
// Max over the 64 lanes of a wave of a non-negative-float bit pattern.  In registers throughout: six exchanges through LDS
// (__shfl_xor) are a chain of 0.3 us, which a kernel of a few rows has nothing to hide under.  With max_of_waves: a row of 4096 quantised
// 2.36 -> 2.04 us, a row of 14336 through SiLU 4.72 -> 4.24, 4096 elements cast with their amax 3.64 -> 3.24, 256 rows of 8192 6.8 -> 5.8.
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
  typedef unsigned pair __attribute__((ext_vector_type(2)));
  v = row_max_u32(v);
  pair s = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  v = s[0] > s[1] ? s[0] : s[1];
  s = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return s[0] > s[1] ? s[0] : s[1];
}
// The largest of a workgroup's waves' values (at most 16 of them, in LDS), in every lane of the calling wave: a loop over them waited
// for LDS once per wave.
__device__ __forceinline__ uint32_t max_of_waves(const uint32_t* parts) {
  const int lane = threadIdx.x & 15;
  return row_max_u32(lane < (int)(blockDim.x >> 6) ? parts[lane] : 0u);
}

}  // namespace mi355q
