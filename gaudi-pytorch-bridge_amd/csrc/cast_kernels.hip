// cast_to_fp8 / cast_from_fp8 / amax kernels for gfx950 and their C entry points.
//
// All three are HBM-bound streaming kernels: every lane moves 16-byte vectors,
// a wave's accesses are contiguous, and each thread keeps several independent
// loads in flight.  Rounding and saturation use the CDNA4 conversion
// instructions (v_cvt_pk_{fp8,bf8}_f32, v_cvt_pk_f32_{fp8,bf8},
// v_cvt_pk_bf16_f32); see device_common.h.
#include <cmath>
#include <type_traits>

#include "device_common.h"

namespace mi355q {

enum ScaleKind { SK_SCALAR = 0, SK_ROW = 1, SK_COL = 2, SK_FULL = 3 };

constexpr int kThreads = 256;

__global__ void fill_u32_kernel(uint32_t* p, uint32_t v) { *p = v; }

// The word that the stream's next call raises to its amax, cleared on the way instead of by a launch of its own.
__device__ __forceinline__ void clear_next(uint32_t* next) {
  if (next != nullptr && blockIdx.x == 0 && threadIdx.x == 0) *next = 0u;
}

// Kernels that reduce an amax run as at most kAmaxBlocks fat workgroups that
// stride over the data: the number of same-address atomics, not the streaming,
// is what bounds them otherwise (2048 blocks: ~30 us; 256 blocks: ~7 us for
// 32 MiB).
constexpr int kAmaxThreads = 1024;
constexpr int kAmaxBlocks = 256;
// The cast with amax: up to kAmaxBlocks workgroups of 512 threads with eight vectors in flight per lane, of 256 threads
// while those suffice (short tensors: more compute units take part).  With the amax starting at zero, bf16, us:
//   elements              2^12   2^20   2^22   2^23   2^24   2^26   2^28
//   this                   4.2    4.5    6.1    7.4   11.4   34.1    131
//   256 x 1024 threads     4.6    5.7    7.3    9.1   11.5   34.9    136
//   up to 2048 x 256       4.3    4.7   11.3   24.6     94     97    154    (atomics on one word: 13 to 45 ns each)
// An fp32 vector is 32 bytes, so four of them are as many bytes as eight of bf16; with eight, and with 1024 threads, fp32, us:
//   elements              2^22   2^23   2^24   2^25   2^26   2^27
//   four, 512 threads      7.5    9.5   17.1   30.8   59.7    118
//   eight, 512 threads     7.9    9.4   18.3   33.8   66.7    134
//   four, 1024 threads     7.8    8.9   17.2   32.0   61.9    123
constexpr int kCastAmaxMaxThreads = 512;
constexpr int cast_amax_vectors(bool bf16_in) { return bf16_in ? 8 : 4; }
constexpr int64_t kCastAmaxSmall = int64_t(1) << 21;  // elements

// Block-level max of abs-value bit patterns, then one atomicMax per block.
// Bit patterns of non-negative floats order like the floats, and a NaN
// pattern is larger than Inf, so NaN wins and the result reads back as NaN.
__device__ __forceinline__ void block_amax_commit(uint32_t m, uint32_t* amax) {
  __shared__ uint32_t wave_part[16];
  m = wave_max_u32(m);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) wave_part[wave] = m;
  __syncthreads();
  if (threadIdx.x >= 64) return;
  const uint32_t r = max_of_waves(wave_part);
  if (threadIdx.x == 0) {
    // Atomics on one address serialise in L2.  The running maximum only grows,
    // so a block whose maximum does not beat the value already there has
    // nothing to add: read it first (device-scope load, not from L1) and skip
    // the atomic.  After the first few blocks almost every block skips.
    if (r != 0 && r > __hip_atomic_load(amax, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(amax, r);
  }
}

// ---------------------------------------------------------------- cast_to_fp8
//
// The input is viewed as [rows, vec_per_row] vectors of 8 elements.  Flat
// modes use rows == 1.  A block owns blockDim*U consecutive vectors of one
// row; U loads per thread are issued before any is consumed.
//   SK_SCALAR  one scale for everything (host value or *scale)
//   SK_ROW     scale[row % mid]
//   SK_COL     scale[column]
//   SK_FULL    scale[element]
//
// The body has no divergent branch: loads and stores go through buffer
// descriptors that cover exactly the block's vectors, so a lane past the end
// of the row loads zeros and its store is dropped.  (With a branch around each
// load the compiler cannot tell that the previous iteration's load into the
// same registers was consumed, and makes every load wait for all earlier ones.)
template <bool BF16_IN, int FMT, int SK, bool AMAX, int U>
__device__ __forceinline__ void cast_to_fp8_vectors(
    const int THREADS,
    const uint8_t* __restrict__ x, uint8_t* __restrict__ y, const float* __restrict__ scale,
    float scale_host, int scale_is_dev, int64_t vec_per_row, int64_t blocks_per_row,
    int64_t total_blocks, int64_t mid, uint32_t* __restrict__ amax, uint32_t* __restrict__ next) {
  constexpr int IN_BYTES = BF16_IN ? 16 : 32;
  constexpr int kNt = 2;  // non-temporal
  uint32_t am = 0;
  if constexpr (AMAX) clear_next(next);
  // a logical block is THREADS * U consecutive vectors of one row; without amax
  // (or with few enough of them) the grid holds one workgroup per logical block and this loop runs once
  for (int64_t lb = blockIdx.x; lb < total_blocks; lb += gridDim.x) {
    const int64_t row = lb / blocks_per_row;
    const int64_t vec0 = (lb - row * blocks_per_row) * (int64_t)(THREADS * U);  // first vector, within the row
    const int64_t left = vec_per_row - vec0;
    const int nvec = (int)(left < THREADS * U ? left : THREADS * U);
    const int64_t first = row * vec_per_row + vec0;                             // first vector, within the tensor
    const __amdgpu_buffer_rsrc_t rin =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(x) + first * IN_BYTES, 0, nvec * IN_BYTES, 0x00020000);
    const __amdgpu_buffer_rsrc_t rout = __builtin_amdgcn_make_buffer_rsrc(y + first * 8, 0, nvec * 8, 0x00020000);

    float s = 1.0f;
    if constexpr (SK == SK_SCALAR) s = scale_is_dev ? scale[0] : scale_host;
    if constexpr (SK == SK_ROW) s = scale[row % mid];
    if constexpr (BF16_IN) s = round_to_bf16(s);

    u32x4 in[U][BF16_IN ? 1 : 2];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int off = ((int)threadIdx.x + u * THREADS) * IN_BYTES;
      in[u][0] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rin, off, 0, kNt));
      if constexpr (!BF16_IN) in[u][1] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rin, off + 16, 0, kNt));
    }
    // per-column / per-element scales: 8 floats per vector, out-of-range lanes read zeros
    u32x4 sc[(SK == SK_COL || SK == SK_FULL) ? U : 1][2];
    if constexpr (SK == SK_COL || SK == SK_FULL) {
      const float* sbase = scale + (SK == SK_COL ? vec0 : first) * 8;
      const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(sbase), 0, nvec * 32, 0x00020000);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int off = ((int)threadIdx.x + u * THREADS) * 32;
        sc[u][0] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0));
        sc[u][1] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, off + 16, 0, 0));
      }
    }

#pragma unroll
    for (int u = 0; u < U; ++u) {
      float v[8];
      if constexpr (BF16_IN) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const uint32_t w = in[u][0][i];
          v[2 * i] = __uint_as_float(w << 16);
          v[2 * i + 1] = __uint_as_float(w & 0xffff0000u);
          if constexpr (AMAX) {
            // packed 16-bit max over the two abs bit patterns of this dword
            const u16x2 a = __builtin_bit_cast(u16x2, w & 0x7fff7fffu);
            const u16x2 m = __builtin_elementwise_max(a, __builtin_bit_cast(u16x2, am));
            am = __builtin_bit_cast(uint32_t, m);
          }
        }
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const uint32_t w = in[u][i >> 2][i & 3];
          v[i] = __uint_as_float(w);
          if constexpr (AMAX) {
            const uint32_t a = w & 0x7fffffffu;
            am = am > a ? am : a;
          }
        }
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        float sv = s;
        if constexpr (SK == SK_COL || SK == SK_FULL) {
          sv = __uint_as_float(sc[u][i >> 2][i & 3]);
          if constexpr (BF16_IN) sv = round_to_bf16(sv);
        }
        float p = v[i] * sv;
        if constexpr (BF16_IN) p = round_to_bf16(p);
        v[i] = p;
      }
      u32x2 out;
      out.x = cvt_fp8x4<FMT>(v[0], v[1], v[2], v[3]);
      out.y = cvt_fp8x4<FMT>(v[4], v[5], v[6], v[7]);
      __builtin_amdgcn_raw_buffer_store_b64(out, rout, ((int)threadIdx.x + u * THREADS) * 8, 0, kNt);
      if constexpr (AMAX) {
        // Where every workgroup has one logical block they all end at once, find the word still at zero and queue up
        // at it.  One wave of each hands in what it has seen halfway, so that most find a larger value at the end and
        // skip (2^22 elements: 6.1 instead of 7.0 us).  Longer tensors spread by themselves and only lose by it.
        if (u == U / 2 - 1 && total_blocks == gridDim.x && threadIdx.x < 64) {
          uint32_t m = am;
          if constexpr (BF16_IN) m = ((m & 0xffffu) > (m >> 16) ? m & 0xffffu : m >> 16) << 16;
          m = wave_max_u32(m);
          if (threadIdx.x == 0) atomicMax(amax, m);
        }
      }
    }
  }

  if constexpr (AMAX) {
    if constexpr (BF16_IN) {
      const uint32_t lo = am & 0xffffu, hi = am >> 16;
      am = (lo > hi ? lo : hi) << 16;
    }
    block_amax_commit(am, amax);
  }
}

template <bool BF16_IN, int FMT, int SK, bool AMAX, int U>
__global__ __launch_bounds__(AMAX ? kCastAmaxMaxThreads : kThreads) void cast_to_fp8_vec8(
    const uint8_t* __restrict__ x, uint8_t* __restrict__ y, const float* __restrict__ scale,
    float scale_host, int scale_is_dev, int64_t vec_per_row, int64_t blocks_per_row,
    int64_t total_blocks, int64_t mid, uint32_t* __restrict__ amax, uint32_t* __restrict__ next) {
  cast_to_fp8_vectors<BF16_IN, FMT, SK, AMAX, U>(AMAX ? (int)blockDim.x : kThreads, x, y, scale, scale_host, scale_is_dev, vec_per_row, blocks_per_row, total_blocks, mid, amax, next);
}

// With amax and rows that hold one or two vectors per thread (cast_amax_shape): less in flight per thread, by design.
template <bool BF16_IN, int FMT, int SK, int U>
__global__ __launch_bounds__(kCastAmaxMaxThreads) void cast_to_fp8_short_rows(
    const uint8_t* __restrict__ x, uint8_t* __restrict__ y, const float* __restrict__ scale, int64_t vec_per_row, int64_t blocks_per_row,
    int64_t total_blocks, int64_t mid, uint32_t* __restrict__ amax, uint32_t* __restrict__ next) {
  cast_to_fp8_vectors<BF16_IN, FMT, SK, true, U>((int)blockDim.x, x, y, scale, 0.0f, 1, vec_per_row, blocks_per_row, total_blocks, mid, amax, next);
}

// Element by element, any alignment, any broadcast: tails and odd shapes.
// A form of its own without amax (with the amax chain's clearing in it, that too, such calls took 6.9 and 11.1 instead of
// 6.4 and 10.2 us, 3001 x 1001 and 16384 x 333 fp32 per column).  With amax a thread takes kGenericAmaxU elements, which
// makes that many fewer workgroups meet at one word: one, four, eight, sixteen elements 22.6, 13.9, 14.4, 12.6 us at
// 3001 x 1001 bf16, 72, 52, 41, 37 at 4095 x 4095, 11.7, 8.3, 7.1, 9.8 at 100 x 3001.
constexpr int kGenericAmaxU = 8;
template <bool BF16_IN, int FMT, bool AMAX>
__global__ __launch_bounds__(kThreads) void cast_to_fp8_generic(
    const uint8_t* __restrict__ x, uint8_t* __restrict__ y, const float* __restrict__ scale,
    float scale_host, int mode, int64_t start, int64_t n, int64_t mid, int64_t inner,
    uint32_t* __restrict__ amax, uint32_t* __restrict__ next) {
  constexpr int U = AMAX ? kGenericAmaxU : 1;
  uint32_t am = 0;
  if constexpr (AMAX) clear_next(next);
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int64_t i = start + ((int64_t)blockIdx.x * U + u) * kThreads + threadIdx.x;
    if (i < n) {
      float s = 1.0f;
      if (mode == MI355Q_SCALE_HOST) s = scale_host;
      else if (mode == MI355Q_SCALE_DEV) s = scale[0];
      else if (mode == MI355Q_SCALE_MID) s = scale[(i / inner) % mid];
      else if (mode == MI355Q_SCALE_FULL) s = scale[i];
      float v, p;
      if constexpr (BF16_IN) {
        const uint32_t h = reinterpret_cast<const uint16_t*>(x)[i];
        v = bf16_bits_to_f32(h);
        p = round_to_bf16(v * round_to_bf16(s));
      } else {
        v = reinterpret_cast<const float*>(x)[i];
        p = v * s;
      }
      const uint32_t a = __float_as_uint(v) & 0x7fffffffu;
      am = am > a ? am : a;
      y[i] = (uint8_t)(cvt_fp8x4<FMT>(p, p, p, p) & 0xffu);
    }
  }
  if constexpr (AMAX) block_amax_commit(am, amax);
}

// Stochastic rounding with flush to zero (round mode CAST_ROUND_SFTZ of GetCastParams,
// hpu_ops/backend/fp8_ops.cpp:105-119): a scaled value below the format's smallest normal number
// becomes a zero of its sign instead of being rounded stochastically among the subnormals.
template <int FMT>
__device__ __forceinline__ float flush_below_min_normal(float p) {
  constexpr float kMinNormal = FMT == MI355Q_E5M2 ? 6.103515625e-05f : 0.015625f;  // 2^-14, 2^-6
  return __builtin_fabsf(p) < kMinNormal ? __builtin_copysignf(0.0f, p) : p;
}

// Stochastic-rounding cast: four consecutive elements per thread, any scale
// broadcast, optional amax.  Not a bandwidth-tuned path (training-side casts of
// optimizer state use it, the inference path rounds to nearest).
template <bool BF16_IN, int FMT>
__global__ __launch_bounds__(kThreads) void cast_to_fp8_sr_kernel(
    const uint8_t* __restrict__ x, uint8_t* __restrict__ y, const float* __restrict__ scale,
    float scale_host, int mode, int64_t n, int64_t mid, int64_t inner, uint64_t seed, uint64_t offset,
    int flush_subnormals, uint32_t* __restrict__ amax) {
  const int64_t q = (int64_t)blockIdx.x * kThreads + threadIdx.x;  // index of this thread's quad
  const int64_t i0 = q * 4;
  uint32_t am = 0;
  if (i0 < n) {
    float p[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int64_t i = i0 + e < n ? i0 + e : n - 1;
      float s = 1.0f;
      if (mode == MI355Q_SCALE_HOST) s = scale_host;
      else if (mode == MI355Q_SCALE_DEV) s = scale[0];
      else if (mode == MI355Q_SCALE_MID) s = scale[(i / inner) % mid];
      else if (mode == MI355Q_SCALE_FULL) s = scale[i];
      float v;
      if constexpr (BF16_IN) {
        v = bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(x)[i]);
        p[e] = round_to_bf16(v * round_to_bf16(s));
      } else {
        v = reinterpret_cast<const float*>(x)[i];
        p[e] = v * s;
      }
      const uint32_t a = __float_as_uint(v) & 0x7fffffffu;
      am = am > a ? am : a;
      if (flush_subnormals) p[e] = flush_below_min_normal<FMT>(p[e]);
    }
    const uint64_t ra = counter_random64(seed, offset + 2 * (uint64_t)q);
    const uint64_t rb = counter_random64(seed, offset + 2 * (uint64_t)q + 1);
    const uint32_t o = cvt_fp8x4_sr<FMT>(p[0], p[1], p[2], p[3], (uint32_t)ra, (uint32_t)(ra >> 32),
                                         (uint32_t)rb, (uint32_t)(rb >> 32));
    if (i0 + 3 < n && (reinterpret_cast<uintptr_t>(y) & 3u) == 0) {
      reinterpret_cast<uint32_t*>(y)[q] = o;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (i0 + e < n) y[i0 + e] = (uint8_t)(o >> (8 * e));
    }
  }
  if (amax != nullptr) block_amax_commit(am, amax);
}

// ------------------------------------------------------------ cast_to_fp8_hybrid
//
// One read of x, two fp8 tensors out (e5m2 with scale_152, e4m3fn with scale_143)
// and optionally amax.  Stochastic rounding applies to the e5m2 output only; the
// e4m3fn output always rounds to nearest even.  Scales are per tensor.
// [first, first + count) elements; VEC = 8 elements per thread per step when the
// pointers allow 16-byte loads, else 1.
template <bool BF16_IN, int VEC>
__global__ __launch_bounds__(kAmaxThreads) void cast_to_fp8_hybrid_kernel(
    const uint8_t* __restrict__ x, uint8_t* __restrict__ y152, uint8_t* __restrict__ y143,
    const float* __restrict__ scale152, const float* __restrict__ scale143, int64_t first, int64_t count,
    int stochastic, uint64_t seed, uint64_t offset, uint32_t* __restrict__ amax) {
  float s5 = scale152 ? scale152[0] : 1.0f, s4 = scale143 ? scale143[0] : 1.0f;
  if constexpr (BF16_IN) {
    s5 = round_to_bf16(s5);
    s4 = round_to_bf16(s4);
  }
  uint32_t am = 0;
  const int64_t steps = (count + VEC - 1) / VEC;
  for (int64_t t = (int64_t)blockIdx.x * kAmaxThreads + threadIdx.x; t < steps; t += (int64_t)gridDim.x * kAmaxThreads) {
    const int64_t i0 = first + t * VEC;
    float v[VEC];
    if constexpr (VEC == 8) {
      if constexpr (BF16_IN) {
        const u32x4 w = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(x + i0 * 2));
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          v[2 * i] = __uint_as_float(w[i] << 16);
          v[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
        }
      } else {
        const f32x4 a = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(x + i0 * 4));
        const f32x4 b = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(x + i0 * 4) + 1);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          v[i] = a[i];
          v[4 + i] = b[i];
        }
      }
    } else {
      v[0] = BF16_IN ? bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(x)[i0]) : reinterpret_cast<const float*>(x)[i0];
    }
    float p5[VEC], p4[VEC];
#pragma unroll
    for (int i = 0; i < VEC; ++i) {
      const uint32_t a = __float_as_uint(v[i]) & 0x7fffffffu;
      am = am > a ? am : a;
      p5[i] = BF16_IN ? round_to_bf16(v[i] * s5) : v[i] * s5;
      p4[i] = BF16_IN ? round_to_bf16(v[i] * s4) : v[i] * s4;
      if (stochastic == 2) p5[i] = flush_below_min_normal<MI355Q_E5M2>(p5[i]);
    }
    if constexpr (VEC == 8) {
      u32x2 o5, o4;
      o4.x = cvt_fp8x4<MI355Q_E4M3FN>(p4[0], p4[1], p4[2], p4[3]);
      o4.y = cvt_fp8x4<MI355Q_E4M3FN>(p4[4], p4[5], p4[6], p4[7]);
      if (stochastic) {
        // element i0 + e draws from counter (i0 + e) / 2, as a scalar step does
        const uint64_t c = offset + (uint64_t)(i0 >> 1);
        const uint64_t r0 = counter_random64(seed, c), r1 = counter_random64(seed, c + 1);
        const uint64_t r2 = counter_random64(seed, c + 2), r3 = counter_random64(seed, c + 3);
        o5.x = cvt_fp8x4_sr<MI355Q_E5M2>(p5[0], p5[1], p5[2], p5[3], (uint32_t)r0, (uint32_t)(r0 >> 32), (uint32_t)r1, (uint32_t)(r1 >> 32));
        o5.y = cvt_fp8x4_sr<MI355Q_E5M2>(p5[4], p5[5], p5[6], p5[7], (uint32_t)r2, (uint32_t)(r2 >> 32), (uint32_t)r3, (uint32_t)(r3 >> 32));
      } else {
        o5.x = cvt_fp8x4<MI355Q_E5M2>(p5[0], p5[1], p5[2], p5[3]);
        o5.y = cvt_fp8x4<MI355Q_E5M2>(p5[4], p5[5], p5[6], p5[7]);
      }
      __builtin_nontemporal_store(o5, reinterpret_cast<u32x2*>(y152 + i0));
      __builtin_nontemporal_store(o4, reinterpret_cast<u32x2*>(y143 + i0));
    } else {
      y143[i0] = (uint8_t)(cvt_fp8x4<MI355Q_E4M3FN>(p4[0], p4[0], p4[0], p4[0]) & 0xffu);
      if (stochastic) {
        const uint64_t r = counter_random64(seed, offset + (uint64_t)(i0 >> 1));
        const uint32_t rr = (i0 & 1) ? (uint32_t)(r >> 32) : (uint32_t)r;
        y152[i0] = (uint8_t)(cvt_fp8x4_sr<MI355Q_E5M2>(p5[0], p5[0], p5[0], p5[0], rr, rr, rr, rr) & 0xffu);
      } else {
        y152[i0] = (uint8_t)(cvt_fp8x4<MI355Q_E5M2>(p5[0], p5[0], p5[0], p5[0]) & 0xffu);
      }
    }
  }
  if (amax != nullptr) block_amax_commit(am, amax);
}

// ---------------------------------------------------------------------- amax
template <bool BF16_IN, int U>
__global__ __launch_bounds__(kAmaxThreads) void amax_vec(const uint8_t* __restrict__ x, int64_t nvec,
                                                         uint32_t* __restrict__ amax) {
  // vectors of 16 bytes; the grid strides over the data
  uint32_t am = 0;
  const int64_t stride = (int64_t)gridDim.x * kAmaxThreads;
  for (int64_t v0 = (int64_t)blockIdx.x * kAmaxThreads + threadIdx.x; v0 < nvec; v0 += stride * U) {
  u32x4 in[U];
  bool ok[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int64_t v = v0 + (int64_t)u * stride;
    ok[u] = v < nvec;
    if (ok[u]) in[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(x) + v);
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (!ok[u]) continue;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (BF16_IN) {
        const u16x2 a = __builtin_bit_cast(u16x2, in[u][i] & 0x7fff7fffu);
        am = __builtin_bit_cast(uint32_t,
                                __builtin_elementwise_max(a, __builtin_bit_cast(u16x2, am)));
      } else {
        const uint32_t a = in[u][i] & 0x7fffffffu;
        am = am > a ? am : a;
      }
    }
  }
  }
  if constexpr (BF16_IN) {
    const uint32_t lo = am & 0xffffu, hi = am >> 16;
    am = (lo > hi ? lo : hi) << 16;
  }
  block_amax_commit(am, amax);
}

template <bool BF16_IN>
__global__ __launch_bounds__(kThreads) void amax_generic(const uint8_t* __restrict__ x,
                                                         int64_t start, int64_t n,
                                                         uint32_t* __restrict__ amax) {
  const int64_t i = start + (int64_t)blockIdx.x * kThreads + threadIdx.x;
  uint32_t am = 0;
  if (i < n) {
    if constexpr (BF16_IN) am = ((uint32_t)reinterpret_cast<const uint16_t*>(x)[i] & 0x7fffu) << 16;
    else am = reinterpret_cast<const uint32_t*>(x)[i] & 0x7fffffffu;
  }
  block_amax_commit(am, amax);
}

// One block per row; rows are independent so no atomics and no pre-zeroing.
template <bool BF16_IN>
__global__ __launch_bounds__(kThreads) void rowwise_amax_kernel(const uint8_t* __restrict__ x,
                                                               int64_t cols, int vec_ok,
                                                               float* __restrict__ out) {
  __shared__ uint32_t wave_part[kThreads / 64];
  const int64_t row = blockIdx.x;
  constexpr int ES = BF16_IN ? 2 : 4;
  const uint8_t* xr = x + row * cols * ES;
  uint32_t am = 0;
  int64_t done = 0;
  if (vec_ok) {
    const int64_t nvec = cols * ES / 16;
    for (int64_t v = threadIdx.x; v < nvec; v += kThreads) {
      const u32x4 w = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(xr) + v);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if constexpr (BF16_IN) {
          const u16x2 a = __builtin_bit_cast(u16x2, w[i] & 0x7fff7fffu);
          am = __builtin_bit_cast(uint32_t,
                                  __builtin_elementwise_max(a, __builtin_bit_cast(u16x2, am)));
        } else {
          const uint32_t a = w[i] & 0x7fffffffu;
          am = am > a ? am : a;
        }
      }
    }
    if constexpr (BF16_IN) {
      const uint32_t lo = am & 0xffffu, hi = am >> 16;
      am = (lo > hi ? lo : hi) << 16;
    }
    done = nvec * (16 / ES);
  }
  for (int64_t c = done + threadIdx.x; c < cols; c += kThreads) {
    uint32_t a;
    if constexpr (BF16_IN) a = ((uint32_t)reinterpret_cast<const uint16_t*>(xr)[c] & 0x7fffu) << 16;
    else a = reinterpret_cast<const uint32_t*>(xr)[c] & 0x7fffffffu;
    am = am > a ? am : a;
  }
  am = wave_max_u32(am);
  if ((threadIdx.x & 63) == 0) wave_part[threadIdx.x >> 6] = am;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t r = wave_part[0];
#pragma unroll
    for (int w = 1; w < kThreads / 64; ++w) r = r > wave_part[w] ? r : wave_part[w];
    out[row] = __uint_as_float(r);
  }
}

// ------------------------------------------------- bf16 rows as two fp8 planes
//
// For the int4-weight GEMM on 16-bit activations (mi355q_w4a16_gemm): a bf16 value has 8 significant
// bits, an e4m3 value 4, so with a power-of-two row scale s (the largest with max |a| s <= 448)
//   hi = e4m3(a s)  (round to nearest even)      lo = e4m3((a s - hi) 16)
// give a s = hi + lo / 16 exactly for every element whose hi is a normal number (the remainder then has
// at most 4 significant bits), and to within 2^-14 (3e-8 of the row's 448) for the small elements whose
// remainder falls below e4m3's subnormal spacing.  The matrix unit multiplies the two planes at the fp8
// rate; 1 / s goes to the GEMM's per-row factor.  One workgroup per row, two passes over it (the second
// out of the cache).  A row of zeros takes s = 1.
__global__ __launch_bounds__(kThreads) void split_rows_kernel(const uint16_t* __restrict__ x, int64_t ldx, int64_t cols,
                                                              uint8_t* __restrict__ hi, uint8_t* __restrict__ lo, int64_t ld,
                                                              float* __restrict__ scale_inv) {
  __shared__ uint32_t wave_part[kThreads / 64];
  const int64_t row = blockIdx.x;
  const uint16_t* xr = x + row * ldx;
  uint32_t am = 0;
  for (int64_t c = threadIdx.x; c < cols; c += kThreads) {
    const uint32_t a = ((uint32_t)xr[c] & 0x7fffu) << 16;
    am = am > a ? am : a;
  }
  am = wave_max_u32(am);
  if ((threadIdx.x & 63) == 0) wave_part[threadIdx.x >> 6] = am;
  __syncthreads();
  uint32_t r = wave_part[0];
#pragma unroll
  for (int w = 1; w < kThreads / 64; ++w) r = r > wave_part[w] ? r : wave_part[w];
  // amax = m 2^ea with 1 <= m < 2; 448 = 1.75 2^8: s = 2^(8 - ea) when m <= 1.75, else 2^(7 - ea)
  int e = 0;
  if (r != 0u && r < 0x7f800000u) {
    const int ea = (int)(r >> 23) - 127;
    e = ((r & 0x007fffffu) <= 0x00600000u ? 8 : 7) - (r >= 0x00800000u ? ea : -126);
    e = e > 126 ? 126 : (e < -126 ? -126 : e);
  }
  const float s = __uint_as_float((uint32_t)(e + 127) << 23);
  if (threadIdx.x == 0) scale_inv[row] = __uint_as_float((uint32_t)(127 - e) << 23);
  uint8_t* hr = hi + row * ld;
  uint8_t* lr = lo + row * ld;
  // four columns per step; ld is a multiple of 16, columns from `cols` to ld are written as zeros
  for (int64_t c = (int64_t)threadIdx.x * 4; c < ld; c += (int64_t)kThreads * 4) {
    float p[4], q[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) p[i] = c + i < cols ? __uint_as_float((uint32_t)xr[c + i] << 16) * s : 0.0f;
    const uint32_t h = cvt_fp8x4<MI355Q_E4M3FN>(p[0], p[1], p[2], p[3]);
    cvt_f32x4<MI355Q_E4M3FN>(h, q[0], q[1], q[2], q[3]);
#pragma unroll
    for (int i = 0; i < 4; ++i) q[i] = (p[i] - q[i]) * 16.0f;   // exact: p and hi agree in their leading bits
    const uint32_t l = cvt_fp8x4<MI355Q_E4M3FN>(q[0], q[1], q[2], q[3]);
    *reinterpret_cast<uint32_t*>(hr + c) = h;
    *reinterpret_cast<uint32_t*>(lr + c) = l;
  }
}

// The same split with the row held in registers (VPT 16-byte vectors of eight bf16 per thread): one pass
// over the row, every load in flight before the first is used, 8-byte stores.  For rows that start 16-byte
// aligned with cols a multiple of 8 and at most 8 * kThreads vectors; output columns from `cols` to ld
// come from lanes whose load falls outside the row's descriptor and reads zeros.  Same bits as the kernel above.
template <int VPT>
__global__ __launch_bounds__(kThreads) void split_rows_vec_kernel(const uint16_t* __restrict__ x, int64_t ldx, int64_t cols,
                                                                  uint8_t* __restrict__ hi, uint8_t* __restrict__ lo, int64_t ld,
                                                                  float* __restrict__ scale_inv) {
  __shared__ uint32_t wave_part[kThreads / 64];
  const int64_t row = blockIdx.x;
  const __amdgpu_buffer_rsrc_t rin = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(x) + row * ldx, 0, (int)cols * 2, 0x00020000);
  const __amdgpu_buffer_rsrc_t rhi = __builtin_amdgcn_make_buffer_rsrc(hi + row * ld, 0, (int)ld, 0x00020000);
  const __amdgpu_buffer_rsrc_t rlo = __builtin_amdgcn_make_buffer_rsrc(lo + row * ld, 0, (int)ld, 0x00020000);
  u32x4 in[VPT];
#pragma unroll
  for (int u = 0; u < VPT; ++u)
    in[u] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rin, ((int)threadIdx.x + u * kThreads) * 16, 0, 0));
  uint32_t am = 0;
#pragma unroll
  for (int u = 0; u < VPT; ++u)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const u16x2 a = __builtin_bit_cast(u16x2, in[u][i] & 0x7fff7fffu);
      am = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(a, __builtin_bit_cast(u16x2, am)));
    }
  {
    const uint32_t l16 = am & 0xffffu, h16 = am >> 16;
    am = (l16 > h16 ? l16 : h16) << 16;
  }
  am = wave_max_u32(am);
  if ((threadIdx.x & 63) == 0) wave_part[threadIdx.x >> 6] = am;
  __syncthreads();
  uint32_t r = wave_part[0];
#pragma unroll
  for (int w = 1; w < kThreads / 64; ++w) r = r > wave_part[w] ? r : wave_part[w];
  int e = 0;
  if (r != 0u && r < 0x7f800000u) {
    const int ea = (int)(r >> 23) - 127;
    e = ((r & 0x007fffffu) <= 0x00600000u ? 8 : 7) - (r >= 0x00800000u ? ea : -126);
    e = e > 126 ? 126 : (e < -126 ? -126 : e);
  }
  const float s = __uint_as_float((uint32_t)(e + 127) << 23);
  if (threadIdx.x == 0) scale_inv[row] = __uint_as_float((uint32_t)(127 - e) << 23);
#pragma unroll
  for (int u = 0; u < VPT; ++u) {
    float p[8], q[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      p[2 * i] = __uint_as_float(in[u][i] << 16) * s;
      p[2 * i + 1] = __uint_as_float(in[u][i] & 0xffff0000u) * s;
    }
    const u32x2 h = {cvt_fp8x4<MI355Q_E4M3FN>(p[0], p[1], p[2], p[3]), cvt_fp8x4<MI355Q_E4M3FN>(p[4], p[5], p[6], p[7])};
    cvt_f32x4<MI355Q_E4M3FN>(h[0], q[0], q[1], q[2], q[3]);
    cvt_f32x4<MI355Q_E4M3FN>(h[1], q[4], q[5], q[6], q[7]);
#pragma unroll
    for (int i = 0; i < 8; ++i) q[i] = (p[i] - q[i]) * 16.0f;
    const u32x2 l = {cvt_fp8x4<MI355Q_E4M3FN>(q[0], q[1], q[2], q[3]), cvt_fp8x4<MI355Q_E4M3FN>(q[4], q[5], q[6], q[7])};
    const int off = ((int)threadIdx.x + u * kThreads) * 8;
    __builtin_amdgcn_raw_buffer_store_b64(h, rhi, off, 0, 0);
    __builtin_amdgcn_raw_buffer_store_b64(l, rlo, off, 0, 0);
  }
}

// Bytes c .. c + 15 of a row of `bytes` bytes that starts anywhere; zeros past its end.  One unaligned 16-byte load: the
// chunk that reaches past the row's end is read so that it ends with the row and shifted into place, so nothing
// outside the row is touched (rows shorter than a chunk: byte by byte).
struct __attribute__((packed, aligned(1))) UnalignedChunk {
  u32x4 v;
};
__device__ __forceinline__ u32x4 ragged_chunk(const uint8_t* row, int c, int bytes) {
  const int n = bytes - c;
  if (bytes < 16) {
    uint32_t w[4] = {0u, 0u, 0u, 0u};
    for (int i = 0; i < n; ++i) w[i >> 2] |= (uint32_t)row[c + i] << (8 * (i & 3));
    return u32x4{w[0], w[1], w[2], w[3]};
  }
  const int back = n < 16 ? 16 - n : 0;
  const u32x4 v = reinterpret_cast<const UnalignedChunk*>(row + c - back)->v;
  if (back == 0) return v;
  const int words = back >> 2, bits = 8 * (back & 3);
  const uint32_t w[8] = {v[0], v[1], v[2], v[3], 0u, 0u, 0u, 0u};
  u32x4 o;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    uint32_t lo = 0u, hi = 0u;
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (k == words) {
        lo = w[i + k];
        hi = w[i + k + 1];
      }
    o[i] = (uint32_t)((((uint64_t)hi << 32) | lo) >> bits);
  }
  return o;
}

// ------------------------------------------------- dynamic per-row quantisation
//
// One pass of "per-row amax -> scale = target / amax -> cast with that scale":
// a workgroup holds one row in registers (VPT 16-byte vectors per thread), so
// the row is read from HBM once.  Results are bit-identical to the three
// separate steps (rowwise_amax, an fp32 division, cast_to_fp8 with per-row
// scales); scale_inv = 1 / scale is what the GEMM takes as A_scale_inv.
//
// A workgroup has as many waves as the row needs (row_shape below): a wave whose lanes are all past the row's end
// would issue the same instructions as the others.  SAT: target's magnitude lies above the largest finite code (or is a
// NaN), so the scaled values need the saturating conversion.
template <int FMT, bool SAT>
__device__ __forceinline__ uint32_t row_cvt_fp8x4(float a, float b, float c, float d) {
  if constexpr (SAT) return cvt_fp8x4<FMT>(a, b, c, d);
  else return cvt_fp8x4_in_range<FMT>(a, b, c, d);
}

constexpr int kMaxRowThreads = 1024;

// The row's amax (a non-negative fp32 bit pattern) from every lane's; then the row's scale, stored by thread 0.
__device__ __forceinline__ float row_scale_of_block(uint32_t am, float target, int64_t row, float* scale_out, float* scale_inv_out) {
  __shared__ uint32_t wave_part[kMaxRowThreads / 64];
  am = wave_max_u32(am);
  if ((threadIdx.x & 63) == 0) wave_part[threadIdx.x >> 6] = am;
  __syncthreads();
  const float scale = row_scale(target, __uint_as_float(max_of_waves(wave_part)));
  if (threadIdx.x == 0) {
    if (scale_out) scale_out[row] = scale;
    if (scale_inv_out) scale_inv_out[row] = 1.0f / scale;
  }
  return scale;
}

template <bool BF16_IN, int FMT, int VPT, bool SAT>
__global__ __launch_bounds__(kMaxRowThreads) void quantize_rows_kernel(
    const uint8_t* __restrict__ x, uint8_t* __restrict__ y, int64_t vec_per_row, float target,
    float* __restrict__ scale_out, float* __restrict__ scale_inv_out) {
  const int64_t row = blockIdx.x;
  const int threads = (int)blockDim.x;
  // Descriptors over the row: a lane past its end loads zeros and its store is
  // dropped, so the body has no divergent branch and all loads are in flight
  // before the first is used.
  constexpr int OUT_BYTES = BF16_IN ? 8 : 4;  // per 16-byte input vector
  const __amdgpu_buffer_rsrc_t rin = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t*>(x) + row * vec_per_row * 16, 0, (int)vec_per_row * 16, 0x00020000);
  const __amdgpu_buffer_rsrc_t rout =
      __builtin_amdgcn_make_buffer_rsrc(y + row * vec_per_row * OUT_BYTES, 0, (int)vec_per_row * OUT_BYTES, 0x00020000);
  u32x4 in[VPT];
  uint32_t am = 0;
#pragma unroll
  for (int u = 0; u < VPT; ++u)
    in[u] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rin, ((int)threadIdx.x + u * threads) * 16, 0, 2));
#pragma unroll
  for (int u = 0; u < VPT; ++u) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (BF16_IN) {
        const u16x2 a = __builtin_bit_cast(u16x2, in[u][i] & 0x7fff7fffu);
        am = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(a, __builtin_bit_cast(u16x2, am)));
      } else {
        const uint32_t a = in[u][i] & 0x7fffffffu;
        am = am > a ? am : a;
      }
    }
  }
  if constexpr (BF16_IN) {
    const uint32_t lo = am & 0xffffu, hi = am >> 16;
    am = (lo > hi ? lo : hi) << 16;
  }
  const float scale = row_scale_of_block(am, target, row, scale_out, scale_inv_out);
  const float s = BF16_IN ? round_to_bf16(scale) : scale;
#pragma unroll
  for (int u = 0; u < VPT; ++u) {
    const int off = ((int)threadIdx.x + u * threads) * OUT_BYTES;
    if constexpr (BF16_IN) {
      float p[8];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        p[2 * i] = round_to_bf16(__uint_as_float(in[u][i] << 16) * s);
        p[2 * i + 1] = round_to_bf16(__uint_as_float(in[u][i] & 0xffff0000u) * s);
      }
      const u32x2 o = {row_cvt_fp8x4<FMT, SAT>(p[0], p[1], p[2], p[3]), row_cvt_fp8x4<FMT, SAT>(p[4], p[5], p[6], p[7])};
      __builtin_amdgcn_raw_buffer_store_b64(o, rout, off, 0, 2);
    } else {
      const uint32_t o = row_cvt_fp8x4<FMT, SAT>(__uint_as_float(in[u][0]) * s, __uint_as_float(in[u][1]) * s,
                                                 __uint_as_float(in[u][2]) * s, __uint_as_float(in[u][3]) * s);
      __builtin_amdgcn_raw_buffer_store_b32(o, rout, off, 0, 2);
    }
  }
}

// The same for rows that are no whole number of vectors or start at any address: unaligned 16-byte loads and 8-byte
// stores, a row's last few codes byte by byte.  (As separate operations, row maxima, division and a cast an element per
// thread, such a call kept the host busy for 28 us.)
template <bool BF16_IN, int FMT>
__global__ __launch_bounds__(kMaxRowThreads) void quantize_ragged_rows_kernel(
    const uint8_t* __restrict__ x, uint8_t* __restrict__ y, int cols, float target,
    float* __restrict__ scale_out, float* __restrict__ scale_inv_out) {
  constexpr int ES = BF16_IN ? 2 : 4, EPV = 16 / ES, VPT = 2;
  const int64_t row = blockIdx.x;
  const int threads = (int)blockDim.x;
  const uint8_t* xr = x + row * cols * ES;
  uint8_t* yr = y + row * cols;
  u32x4 in[VPT];
  uint32_t am = 0;
#pragma unroll
  for (int u = 0; u < VPT; ++u) {
    const int e = ((int)threadIdx.x + u * threads) * EPV;
    in[u] = e < cols ? ragged_chunk(xr, e * ES, cols * ES) : u32x4{0u, 0u, 0u, 0u};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t w = in[u][i];
      const uint32_t a = BF16_IN ? (w << 16) & 0x7fffffffu : w & 0x7fffffffu, b = BF16_IN ? w & 0x7fff0000u : 0u;
      am = am > a ? am : a;
      am = am > b ? am : b;
    }
  }
  const float scale = row_scale_of_block(am, target, row, scale_out, scale_inv_out);
  const float s = BF16_IN ? round_to_bf16(scale) : scale;
#pragma unroll
  for (int u = 0; u < VPT; ++u) {
    const int e = ((int)threadIdx.x + u * threads) * EPV, n = cols - e;
    if (n <= 0) continue;
    float p[EPV];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (BF16_IN) {
        p[2 * i] = round_to_bf16(__uint_as_float(in[u][i] << 16) * s);
        p[2 * i + 1] = round_to_bf16(__uint_as_float(in[u][i] & 0xffff0000u) * s);
      } else {
        p[i] = __uint_as_float(in[u][i]) * s;
      }
    }
    uint32_t o[EPV / 4];
#pragma unroll
    for (int i = 0; i < EPV / 4; ++i) o[i] = cvt_fp8x4<FMT>(p[4 * i], p[4 * i + 1], p[4 * i + 2], p[4 * i + 3]);
    if (n >= EPV) {
      __builtin_memcpy(yr + e, o, EPV);
    } else {
      for (int i = 0; i < n; ++i) yr[e + i] = (uint8_t)(o[i >> 2] >> (8 * (i & 3)));
    }
  }
}

// SiLU(gate) * up in bf16 followed by the dynamic per-row quantisation above,
// in one pass: bf16(bf16(silu(gate)) * up), row amax of that, scale = target /
// amax, cast.  The glue between the gate / up projections and the down
// projection of a decoder MLP block; gate and up may be column ranges of one
// wider matrix (row pitches ld_gate, ld_up in elements).  h_out, when given,
// receives the bf16 products.
//
// Bound by vector issue where the chip is full and by one compute unit's where there is one row, hence the spelling of
// silu_for_bf16 and the maximum over the unrounded products (rounding is monotonic, so the largest rounded product is
// the rounded largest product; the maximum passes a NaN on).  1 x 14336: 4.8 us (7.5 with an IEEE exponential and
// division per element), 1024 x 14336: 14.9 (22.7), 4096 x 14336: 51 us, 5.8 TB/s (60 with bf16(silu) looked up in a
// table in LDS that every workgroup built).
template <int FMT, int VPT, bool SAT>
__global__ __launch_bounds__(kMaxRowThreads) void silu_mul_quantize_rows_kernel(
    const uint16_t* __restrict__ gate, int64_t ld_gate, const uint16_t* __restrict__ up, int64_t ld_up,
    uint8_t* __restrict__ y, uint16_t* __restrict__ h_out, int64_t vec_per_row, float target,
    float* __restrict__ scale_out, float* __restrict__ scale_inv_out) {
  const int64_t row = blockIdx.x;
  const int threads = (int)blockDim.x;
  // Descriptors over the row (zeros past its end, stores dropped there): no
  // divergent branch, and every load is in flight before the first is used.
  const int row_bytes = (int)vec_per_row * 16;
  const __amdgpu_buffer_rsrc_t rg = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(gate) + row * ld_gate, 0, row_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t ru = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(up) + row * ld_up, 0, row_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rh = __builtin_amdgcn_make_buffer_rsrc(
      h_out ? h_out + row * vec_per_row * 8 : nullptr, 0, h_out ? row_bytes : 0, 0x00020000);
  const __amdgpu_buffer_rsrc_t rout = __builtin_amdgcn_make_buffer_rsrc(y + row * vec_per_row * 8, 0, (int)vec_per_row * 8, 0x00020000);
  u32x4 gv[VPT], h[VPT];
  float am = 0.0f;
#pragma unroll
  for (int u = 0; u < VPT; ++u) {
    const int off = ((int)threadIdx.x + u * threads) * 16;
    gv[u] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rg, off, 0, 2));
    h[u] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(ru, off, 0, 2));
  }
#pragma unroll
  for (int u = 0; u < VPT; ++u) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t s = pack_bf16x2(silu_for_bf16(__uint_as_float(gv[u][i] << 16)), silu_for_bf16(__uint_as_float(gv[u][i] & 0xffff0000u)));
      const float h0 = __uint_as_float(s << 16) * __uint_as_float(h[u][i] << 16);
      const float h1 = __uint_as_float(s & 0xffff0000u) * __uint_as_float(h[u][i] & 0xffff0000u);
      am = __builtin_elementwise_maximum(__builtin_elementwise_maximum(__builtin_fabsf(h0), __builtin_fabsf(h1)), am);
      h[u][i] = pack_bf16x2(h0, h1);
    }
    // without h_out the descriptor is empty and the store goes nowhere
    __builtin_amdgcn_raw_buffer_store_b128(h[u], rh, ((int)threadIdx.x + u * threads) * 16, 0, 0);
  }
  const float scale = row_scale_of_block(__float_as_uint(round_to_bf16(am)) & 0x7fffffffu, target, row, scale_out, scale_inv_out);
  const float s = round_to_bf16(scale);
#pragma unroll
  for (int u = 0; u < VPT; ++u) {
    float p[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      p[2 * i] = round_to_bf16(__uint_as_float(h[u][i] << 16) * s);
      p[2 * i + 1] = round_to_bf16(__uint_as_float(h[u][i] & 0xffff0000u) * s);
    }
    const u32x2 o = {row_cvt_fp8x4<FMT, SAT>(p[0], p[1], p[2], p[3]), row_cvt_fp8x4<FMT, SAT>(p[4], p[5], p[6], p[7])};
    __builtin_amdgcn_raw_buffer_store_b64(o, rout, ((int)threadIdx.x + u * threads) * 8, 0, 2);
  }
}

// -------------------------------------------------------------- cast_from_fp8
//
// A lane produces one 16-byte store: 8 fp8 bytes in for bf16 output, 4 for
// fp32 output.  A wave's store then covers 1 KiB of whole cache lines; wider
// loads would leave each lane with several stores that each touch only part
// of a line, and those partial-line writes cost HBM bandwidth.
template <bool BF16_OUT>
constexpr int from_vec() { return BF16_OUT ? 8 : 4; }

// WINDOW: stores a wave may still have outstanding when it issues the next one
// (-1: no limit).  Measured for bf16 output, which writes twice the bytes it
// reads: with 2 the kernel is 3-8 % faster than unlimited from 64 MiB of output
// up (6.2 TB/s at 512 MiB), with 0 it is 9 % faster at 32 MiB; other sizes do
// not care.  fp32 output and cast_to_fp8 (more reads than writes) lose with any limit.
template <int FMT, bool BF16_OUT, int SK, int U, int WINDOW>
__global__ __launch_bounds__(kThreads) void cast_from_fp8_vec(
    const uint8_t* __restrict__ x, uint8_t* __restrict__ y, const float* __restrict__ scale,
    float scale_host, int scale_is_dev, int has_scale, int64_t vec_per_row,
    int64_t blocks_per_row, int64_t mid) {
  constexpr int V = from_vec<BF16_OUT>();
  constexpr int kNt = 2;  // non-temporal
  const int64_t row = blockIdx.x / blocks_per_row;
  const int64_t vec0 = (blockIdx.x - row * blocks_per_row) * (int64_t)(kThreads * U);  // first vector, within the row
  const int64_t left = vec_per_row - vec0;
  const int nvec = (int)(left < kThreads * U ? left : kThreads * U);
  const int64_t first = row * vec_per_row + vec0;                                    // first vector, within the tensor
  // Branch-free like cast_to_fp8_vec8: descriptors that cover the block's
  // vectors make a lane past the end load zeros and drop its store.
  const __amdgpu_buffer_rsrc_t rin = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(x) + first * V, 0, nvec * V, 0x00020000);
  const __amdgpu_buffer_rsrc_t rout = __builtin_amdgcn_make_buffer_rsrc(y + first * 16, 0, nvec * 16, 0x00020000);

  float s = 1.0f;
  if constexpr (SK == SK_SCALAR) s = scale_is_dev ? scale[0] : scale_host;
  if constexpr (SK == SK_ROW) s = scale[row % mid];
  if constexpr (BF16_OUT) s = round_to_bf16(s);
  if (!has_scale) s = 1.0f;  // x * 1 == x bit for bit (NaN payloads aside, and fp8 NaNs have one)

  uint32_t in[U][V / 4];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int off = ((int)threadIdx.x + u * kThreads) * V;
    if constexpr (V == 8) {
      const u32x2 t = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rin, off, 0, kNt));
      in[u][0] = t[0];
      in[u][1] = t[1];
    } else {
      in[u][0] = __builtin_amdgcn_raw_buffer_load_b32(rin, off, 0, kNt);
    }
  }
  constexpr bool kVecScale = SK == SK_COL || SK == SK_FULL;
  u32x4 sc[kVecScale ? U : 1][V / 4];
  if constexpr (kVecScale) {  // the launcher picks these kinds only for a scale tensor
    const float* sbase = scale + (SK == SK_COL ? vec0 : first) * V;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(sbase), 0, nvec * V * 4, 0x00020000);
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int q = 0; q < V / 4; ++q)
        sc[u][q] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, ((int)threadIdx.x + u * kThreads) * V * 4 + 16 * q, 0, 0));
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    float v[V];
#pragma unroll
    for (int i = 0; i < V / 4; ++i)
      cvt_f32x4<FMT>(in[u][i], v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]);
#pragma unroll
    for (int i = 0; i < V; ++i) {
      float sv = s;
      if constexpr (kVecScale) {
        sv = __uint_as_float(sc[u][i >> 2][i & 3]);
        if constexpr (BF16_OUT) sv = round_to_bf16(sv);
      }
      v[i] *= sv;
    }
    u32x4 t;
    if constexpr (BF16_OUT) {
#pragma unroll
      for (int i = 0; i < 4; ++i) t[i] = pack_bf16x2(v[2 * i], v[2 * i + 1]);
    } else {
      t = u32x4{__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3])};
    }
    __builtin_amdgcn_raw_buffer_store_b128(t, rout, ((int)threadIdx.x + u * kThreads) * 16, 0, kNt);
    if constexpr (WINDOW >= 0) {
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_waitcnt(0x0F70 | WINDOW);  // vmcnt(WINDOW), other counters unlimited
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

template <int FMT, bool BF16_OUT>
__global__ __launch_bounds__(kThreads) void cast_from_fp8_generic(
    const uint8_t* __restrict__ x, uint8_t* __restrict__ y, const float* __restrict__ scale,
    float scale_host, int mode, int64_t start, int64_t n, int64_t mid, int64_t inner) {
  const int64_t i = start + (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (i >= n) return;
  float v = cvt_f32x1<FMT>(x[i]);
  if (mode != MI355Q_SCALE_NONE) {
    float s = 1.0f;
    if (mode == MI355Q_SCALE_HOST) s = scale_host;
    else if (mode == MI355Q_SCALE_DEV) s = scale[0];
    else if (mode == MI355Q_SCALE_MID) s = scale[(i / inner) % mid];
    else if (mode == MI355Q_SCALE_FULL) s = scale[i];
    if constexpr (BF16_OUT) s = round_to_bf16(s);
    v *= s;
  }
  if constexpr (BF16_OUT) reinterpret_cast<uint16_t*>(y)[i] = (uint16_t)(pack_bf16x2(v, v) & 0xffffu);
  else reinterpret_cast<float*>(y)[i] = v;
}

__global__ __launch_bounds__(kThreads) void copy_bytes_kernel(const uint8_t* __restrict__ x,
                                                              uint8_t* __restrict__ y, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (i < n) y[i] = x[i];
}

constexpr int kCopyU = 4;  // 16-byte vectors per thread

// A block copies kThreads * kCopyU vectors through descriptors that end with
// the tensor: all loads of a lane are issued before its first store.
__global__ __launch_bounds__(kThreads) void copy_vec16_kernel(const uint8_t* __restrict__ x,
                                                              uint8_t* __restrict__ y, int64_t nvec) {
  const int64_t v0 = (int64_t)blockIdx.x * (kThreads * kCopyU);
  const int64_t left = nvec - v0;
  const int bytes = (int)(left < kThreads * kCopyU ? left : kThreads * kCopyU) * 16;
  const __amdgpu_buffer_rsrc_t rin = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(x) + v0 * 16, 0, bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rout = __builtin_amdgcn_make_buffer_rsrc(y + v0 * 16, 0, bytes, 0x00020000);
  u32x4 t[kCopyU];
#pragma unroll
  for (int u = 0; u < kCopyU; ++u)
    t[u] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rin, ((int)threadIdx.x + u * kThreads) * 16, 0, 2));
#pragma unroll
  for (int u = 0; u < kCopyU; ++u)
    __builtin_amdgcn_raw_buffer_store_b128(t[u], rout, ((int)threadIdx.x + u * kThreads) * 16, 0, 2);
}

// ------------------------------------------------------------- padded copies
//
// Byte matrices whose rows start at any address, copied into rows of whole 16-byte chunks with zeros behind the data
// (what the GEMM's MFMA kernels take): both operands of a product in one launch.  A thread writes kPadU chunks of the
// destination and reads each with one unaligned 16-byte load; the last chunk of a row is read so that it ends with
// the row and shifted into place, so nothing outside the matrix is touched.
struct PadJob {
  const uint8_t* src;
  uint8_t* dst;
  int64_t src_ld, src_stride, dst_stride;  // bytes
  int32_t rows, cols, dst_rows, dst_chunks;
  int32_t batch;
  int64_t chunks;                          // of all matrices
};
struct PadJobs {
  PadJob job[2];
};
constexpr int kPadU = 4;

// The chunk `k` chunks behind the start of row `row0` (of all matrices' rows).
__device__ __forceinline__ u32x4 pad_chunk(const PadJob& j, int64_t row0, uint32_t k) {
  const uint32_t down = k / (uint32_t)j.dst_chunks;
  const int c = (int)(k - down * (uint32_t)j.dst_chunks) * 16;
  const int64_t row_all = row0 + down;
  int64_t b = 0, r = row_all;
  if (j.batch > 1) {
    b = row_all / j.dst_rows;
    r = row_all - b * j.dst_rows;
  }
  if (r >= j.rows || c >= j.cols) return u32x4{0u, 0u, 0u, 0u};
  return ragged_chunk(j.src + b * j.src_stride + r * j.src_ld, c, j.cols);
}

__global__ __launch_bounds__(kThreads) void pad_rows_kernel(PadJobs jobs, int64_t blocks0) {
  const bool second = blockIdx.x >= blocks0;
  const PadJob& j = jobs.job[second ? 1 : 0];
  const int64_t start = ((int64_t)blockIdx.x - (second ? blocks0 : 0)) * (kThreads * kPadU), first = start + threadIdx.x;
  const int64_t row0 = start / j.dst_chunks;
  const uint32_t k0 = (uint32_t)(start - row0 * j.dst_chunks) + threadIdx.x;
  u32x4 v[kPadU];
#pragma unroll
  for (int u = 0; u < kPadU; ++u)
    v[u] = first + u * kThreads < j.chunks ? pad_chunk(j, row0, k0 + u * kThreads) : u32x4{0u, 0u, 0u, 0u};
#pragma unroll
  for (int u = 0; u < kPadU; ++u) {
    const int64_t chunk = first + u * kThreads;
    if (chunk < j.chunks) *reinterpret_cast<u32x4*>(j.dst + chunk * 16) = v[u];
  }
}

// --------------------------------------------------------------- host helpers

inline bool aligned(const void* p, size_t a) { return (reinterpret_cast<uintptr_t>(p) % a) == 0; }
inline int launch_status() { return hipGetLastError() == hipSuccess ? MI355Q_OK : MI355Q_ERR_LAUNCH; }
inline unsigned blocks_for(int64_t n, int64_t per) { return (unsigned)((n + per - 1) / per); }

// Decide how the vector kernels see the problem.  Returns false when only the
// generic kernel applies.
struct VecPlan {
  int sk;
  int64_t rows, row_len, mid;
};

inline bool plan_vectors(int mode, int64_t outer, int64_t mid, int64_t inner, int64_t vec,
                         VecPlan* p) {
  const int64_t n = outer * mid * inner;
  switch (mode) {
    case MI355Q_SCALE_NONE:
    case MI355Q_SCALE_HOST:
    case MI355Q_SCALE_DEV:
      *p = {SK_SCALAR, 1, n, 1};
      return true;
    case MI355Q_SCALE_FULL:
      *p = {SK_FULL, 1, n, 1};
      return true;
    case MI355Q_SCALE_MID:
      if (inner == 1) {  // per column of [outer, mid]
        if (mid % vec != 0 || mid < 4 * vec) return false;
        *p = {SK_COL, outer, mid, mid};
        return true;
      }
      if (inner % vec != 0 || inner < 4 * vec) return false;
      *p = {SK_ROW, outer * mid, inner, mid};
      return true;
    default:
      return false;
  }
}

constexpr int kCastU = 4;  // 16-byte loads in flight per thread

// How a cast with amax runs: threads of a workgroup, and vectors in flight per thread.  Where rows have scales of their own, or
// columns have, a workgroup walks row by row and a thread has no more vectors to ask for than the row holds: eight at a
// time would be empty steps and, with the amax kernels' few workgroups, little in flight.  bf16, us, with 8 and with this:
//   4096 x 4096 per column 52 -> 17 (46 as 1024 threads x 4), per row 41 -> 17 (38)     512 x 16384 per column 10.8 -> 7.8 (9.6)
//   16384 x 64 per column 110 -> 35 (157)     4096 x 512 per column 29 -> 9 (42)     256 x 4096 per column 6.6 -> 4.1 (7.5)
struct CastAmaxShape {
  unsigned threads;
  int vectors;
};
template <bool BF16_IN>
CastAmaxShape cast_amax_shape(int sk, int64_t rows, int64_t vpr) {
  const bool small = rows * vpr * 8 <= kCastAmaxSmall;
  const unsigned threads = small ? kThreads : kCastAmaxMaxThreads;
  if (sk == SK_SCALAR || sk == SK_FULL) return {threads, cast_amax_vectors(BF16_IN)};
  return {threads, small || vpr <= kCastAmaxMaxThreads ? 1 : (vpr <= 2 * kCastAmaxMaxThreads ? 2 : (vpr <= 4 * kCastAmaxMaxThreads ? 4 : cast_amax_vectors(BF16_IN)))};
}

template <bool BF16_IN, int FMT, bool AMAX, int U>
void launch_cast_to_rows(int sk, hipStream_t st, const uint8_t* x, uint8_t* y, const float* scale, int64_t vpr, int64_t bpr,
                         int64_t total, int64_t mid, unsigned threads, uint32_t* amax, uint32_t* next) {
  const unsigned grid = (unsigned)(AMAX && total > kAmaxBlocks ? kAmaxBlocks : total);
  if constexpr (U < 4) {
    if (sk == SK_ROW) cast_to_fp8_short_rows<BF16_IN, FMT, SK_ROW, U><<<grid, threads, 0, st>>>(x, y, scale, vpr, bpr, total, mid, amax, next);
    else cast_to_fp8_short_rows<BF16_IN, FMT, SK_COL, U><<<grid, threads, 0, st>>>(x, y, scale, vpr, bpr, total, mid, amax, next);
  } else if (sk == SK_ROW) {
    cast_to_fp8_vec8<BF16_IN, FMT, SK_ROW, AMAX, U><<<grid, threads, 0, st>>>(x, y, scale, 0.0f, 1, vpr, bpr, total, mid, amax, next);
  } else {
    cast_to_fp8_vec8<BF16_IN, FMT, SK_COL, AMAX, U><<<grid, threads, 0, st>>>(x, y, scale, 0.0f, 1, vpr, bpr, total, mid, amax, next);
  }
}

template <bool BF16_IN, int FMT, bool AMAX>
void launch_cast_to_vec(int sk, hipStream_t st, const uint8_t* x, uint8_t* y, const float* scale, float sh, int is_dev, int64_t vpr,
                        int64_t bpr, int64_t total, int64_t mid, CastAmaxShape shape, uint32_t* amax, uint32_t* next) {
  constexpr int U = AMAX ? cast_amax_vectors(BF16_IN) : kCastU;
  const unsigned T = AMAX ? shape.threads : kThreads;
  const unsigned grid = (unsigned)(AMAX && total > kAmaxBlocks ? kAmaxBlocks : total);
  if (sk == SK_SCALAR) {
    cast_to_fp8_vec8<BF16_IN, FMT, SK_SCALAR, AMAX, U><<<grid, T, 0, st>>>(x, y, scale, sh, is_dev, vpr, bpr, total, mid, amax, next);
  } else if (sk == SK_FULL) {
    cast_to_fp8_vec8<BF16_IN, FMT, SK_FULL, AMAX, U><<<grid, T, 0, st>>>(x, y, scale, sh, is_dev, vpr, bpr, total, mid, amax, next);
  } else if constexpr (!AMAX) {
    launch_cast_to_rows<BF16_IN, FMT, AMAX, U>(sk, st, x, y, scale, vpr, bpr, total, mid, T, amax, next);
  } else {
    switch (shape.vectors) {
      case 1: launch_cast_to_rows<BF16_IN, FMT, AMAX, 1>(sk, st, x, y, scale, vpr, bpr, total, mid, T, amax, next); break;
      case 2: launch_cast_to_rows<BF16_IN, FMT, AMAX, 2>(sk, st, x, y, scale, vpr, bpr, total, mid, T, amax, next); break;
      case 4: launch_cast_to_rows<BF16_IN, FMT, AMAX, 4>(sk, st, x, y, scale, vpr, bpr, total, mid, T, amax, next); break;
      default: launch_cast_to_rows<BF16_IN, FMT, AMAX, U>(sk, st, x, y, scale, vpr, bpr, total, mid, T, amax, next); break;
    }
  }
}

template <bool BF16_IN, int FMT>
int cast_to_dispatch(const uint8_t* x, uint8_t* y, const float* scale, float sh, int mode,
                     int64_t outer, int64_t mid, int64_t inner, uint32_t* amax, uint32_t* next, hipStream_t st) {
  const int64_t n = outer * mid * inner;
  VecPlan p;
  const bool vec = aligned(x, 16) && aligned(y, 8) &&
                   (scale == nullptr || aligned(scale, 16)) && plan_vectors(mode, outer, mid, inner, 8, &p);
  int64_t done = 0;
  if (vec) {
    const int64_t vpr = p.row_len / 8;
    // In flat modes the row length need not be a multiple of 8: the tail goes
    // to the generic kernel.  In 2-D modes plan_vectors has required it.
    if (vpr > 0) {
      const CastAmaxShape shape = cast_amax_shape<BF16_IN>(p.sk, p.rows, vpr);
      const int64_t per_block = amax ? (int64_t)shape.threads * shape.vectors : (int64_t)kThreads * kCastU;
      const int64_t bpr = (vpr + per_block - 1) / per_block;
      const int64_t total = bpr * p.rows;
      if (total > 0x7fffffffLL) return MI355Q_ERR_UNSUPPORTED;
      const int is_dev = mode == MI355Q_SCALE_DEV;
      if (amax) launch_cast_to_vec<BF16_IN, FMT, true>(p.sk, st, x, y, scale, sh, is_dev, vpr, bpr, total, p.mid, shape, amax, next);
      else launch_cast_to_vec<BF16_IN, FMT, false>(p.sk, st, x, y, scale, sh, is_dev, vpr, bpr, total, p.mid, shape, amax, next);
      done = p.rows == 1 ? vpr * 8 : n;
    }
  }
  if (done < n) {
    const int64_t rest = n - done;
    const int64_t per_block = (int64_t)kThreads * (amax ? kGenericAmaxU : 1), grid = (rest + per_block - 1) / per_block;
    if (grid > 0x7fffffffLL) return MI355Q_ERR_UNSUPPORTED;
    if (amax) cast_to_fp8_generic<BF16_IN, FMT, true><<<(unsigned)grid, kThreads, 0, st>>>(x, y, scale, sh, mode, done, n, mid, inner, amax, done > 0 ? nullptr : next);
    else cast_to_fp8_generic<BF16_IN, FMT, false><<<(unsigned)grid, kThreads, 0, st>>>(x, y, scale, sh, mode, done, n, mid, inner, nullptr, nullptr);
  }
  return launch_status();
}

template <int FMT, bool BF16_OUT>
int cast_from_dispatch(const uint8_t* x, uint8_t* y, const float* scale, float sh, int mode,
                       int64_t outer, int64_t mid, int64_t inner, hipStream_t st) {
  constexpr int U = 4;
  constexpr int V = from_vec<BF16_OUT>();
  const int64_t n = outer * mid * inner;
  VecPlan p;
  const bool vec = aligned(x, V) && aligned(y, 16) &&
                   (scale == nullptr || aligned(scale, 16)) && plan_vectors(mode, outer, mid, inner, V, &p);
  int64_t done = 0;
  if (vec) {
    const int64_t vpr = p.row_len / V;
    if (vpr > 0) {
      const int64_t bpr = (vpr + kThreads * U - 1) / (kThreads * U);
      const int64_t grid64 = bpr * p.rows;
      if (grid64 > 0x7fffffffLL) return MI355Q_ERR_UNSUPPORTED;
      const unsigned grid = (unsigned)grid64;
      const int is_dev = mode == MI355Q_SCALE_DEV;
      const int has_scale = mode != MI355Q_SCALE_NONE;
      auto launch = [&](auto window) {
        constexpr int W = decltype(window)::value;
        switch (p.sk) {
          case SK_SCALAR:
            cast_from_fp8_vec<FMT, BF16_OUT, SK_SCALAR, U, W><<<grid, kThreads, 0, st>>>(x, y, scale, sh, is_dev, has_scale, vpr, bpr, p.mid);
            break;
          case SK_ROW:
            cast_from_fp8_vec<FMT, BF16_OUT, SK_ROW, U, W><<<grid, kThreads, 0, st>>>(x, y, scale, sh, is_dev, has_scale, vpr, bpr, p.mid);
            break;
          case SK_COL:
            cast_from_fp8_vec<FMT, BF16_OUT, SK_COL, U, W><<<grid, kThreads, 0, st>>>(x, y, scale, sh, is_dev, has_scale, vpr, bpr, p.mid);
            break;
          default:
            cast_from_fp8_vec<FMT, BF16_OUT, SK_FULL, U, W><<<grid, kThreads, 0, st>>>(x, y, scale, sh, is_dev, has_scale, vpr, bpr, p.mid);
            break;
        }
      };
      if constexpr (BF16_OUT) {
        if (n * 2 <= (int64_t(48) << 20)) launch(std::integral_constant<int, 0>{});
        else launch(std::integral_constant<int, 2>{});
      } else {
        launch(std::integral_constant<int, -1>{});
      }
      done = p.rows == 1 ? vpr * V : n;
    }
  }
  if (done < n) {
    const int64_t grid = (n - done + kThreads - 1) / kThreads;
    if (grid > 0x7fffffffLL) return MI355Q_ERR_UNSUPPORTED;
    cast_from_fp8_generic<FMT, BF16_OUT><<<(unsigned)grid, kThreads, 0, st>>>(x, y, scale, sh, mode, done, n, mid, inner);
  }
  return launch_status();
}

inline bool scale_args_ok(const float* scale, int mode, int64_t outer, int64_t mid, int64_t inner) {
  if (mode < MI355Q_SCALE_NONE || mode > MI355Q_SCALE_FULL) return false;
  if (outer < 0 || mid < 0 || inner < 0) return false;
  if ((mode == MI355Q_SCALE_DEV || mode == MI355Q_SCALE_MID || mode == MI355Q_SCALE_FULL) && scale == nullptr)
    return false;
  return true;
}

// How a row of vpr vectors is spread over a workgroup: vectors per thread, and threads, whole waves of them.
// Few rows leave compute units idle, and a row's time is that of its slowest thread: one vector per thread, two where
// 1024 threads do not suffice.  With many rows four vectors per thread keep more loads in flight and several
// workgroups on a compute unit (three, five or seven: 3 to 10 % slower at 1024 x 14336 and 2048 x 5632; at 512 rows
// the two forms cross).  Rows of more than 2048 vectors (the inner width of a 70B-class MLP) have four per thread at any
// number of rows; as separate operations (aten's silu and mul, row maxima, a division, a cast, a reciprocal) 4 x 19904
// took nine launches, and the whole MLP of 4 x 7488 / 19904 114 us against 98 with one kernel.
constexpr int64_t kFewRows = 512;
constexpr int kBulkVectors = 4;
struct RowShape {
  int vpt;
  unsigned threads;
};
inline RowShape row_shape(int64_t rows, int64_t vpr) {
  const int vpt = rows < kFewRows && vpr <= 2 * kMaxRowThreads ? (vpr <= kMaxRowThreads ? 1 : 2) : kBulkVectors;
  return {vpt, (unsigned)(((vpr + vpt - 1) / vpt + 63) / 64 * 64)};
}
constexpr int64_t kMaxRowVectors = kBulkVectors * kMaxRowThreads, kMaxRaggedVectors = 2 * kMaxRowThreads;

// Calls f(vectors per thread, saturate, threads); false: the row does not fit a workgroup.
template <int FMT, typename F>
bool with_row_shape(int64_t rows, int64_t vpr, float target, F&& f) {
  if (vpr > kMaxRowVectors) return false;
  const RowShape s = row_shape(rows, vpr);
  auto with_vectors = [&](auto saturate) {
    if (s.vpt == 1) f(std::integral_constant<int, 1>{}, saturate, s.threads);
    else if (s.vpt == 2) f(std::integral_constant<int, 2>{}, saturate, s.threads);
    else f(std::integral_constant<int, kBulkVectors>{}, saturate, s.threads);
  };
  // (both conversions with the same shapes: a saturating form with 1024 threads for every row took 23 instead of 7 us at
  // 4096 x 1024 and 45 instead of 8 at 8192 x 512)
  if (!(std::fabs(target) <= kFp8Max[FMT - MI355Q_E4M3FN])) with_vectors(std::true_type{});
  else with_vectors(std::false_type{});
  return true;
}

template <bool BF16_IN, int FMT>
int quantize_rows_launch(const uint8_t* x, uint8_t* y, int64_t rows, int64_t vpr, float target,
                         float* scale_out, float* scale_inv_out, hipStream_t st) {
  const bool ok = with_row_shape<FMT>(rows, vpr, target, [&](auto v, auto sat, unsigned threads) {
    quantize_rows_kernel<BF16_IN, FMT, decltype(v)::value, decltype(sat)::value>
        <<<(unsigned)rows, threads, 0, st>>>(x, y, vpr, target, scale_out, scale_inv_out);
  });
  return ok ? launch_status() : MI355Q_ERR_UNSUPPORTED;
}

template <int FMT>
int silu_mul_quantize_rows_launch(const uint16_t* gate, int64_t ld_gate, const uint16_t* up, int64_t ld_up,
                                  uint8_t* y, uint16_t* h_out, int64_t rows, int64_t vpr, float target,
                                  float* scale_out, float* scale_inv_out, hipStream_t st) {
  const bool ok = with_row_shape<FMT>(rows, vpr, target, [&](auto v, auto sat, unsigned threads) {
    silu_mul_quantize_rows_kernel<FMT, decltype(v)::value, decltype(sat)::value>
        <<<(unsigned)rows, threads, 0, st>>>(gate, ld_gate, up, ld_up, y, h_out, vpr, target, scale_out, scale_inv_out);
  });
  return ok ? launch_status() : MI355Q_ERR_UNSUPPORTED;
}

}  // namespace mi355q

using namespace mi355q;

extern "C" {

int mi355q_amax(const void* x, int x_dtype, int64_t n, float* amax_out, void* stream) {
  if (amax_out == nullptr || n < 0 || (n > 0 && x == nullptr)) return MI355Q_ERR_INVALID_ARGUMENT;
  if (x_dtype != MI355Q_F32 && x_dtype != MI355Q_BF16) return MI355Q_ERR_INVALID_ARGUMENT;
  hipStream_t st = static_cast<hipStream_t>(stream);
  uint32_t* am = reinterpret_cast<uint32_t*>(amax_out);
  fill_u32_kernel<<<1, 1, 0, st>>>(am, 0u);
  if (n == 0) return launch_status();
  constexpr int U = 4;
  const int es = x_dtype == MI355Q_BF16 ? 2 : 4;
  const uint8_t* xb = static_cast<const uint8_t*>(x);
  int64_t done = 0;
  if (aligned(x, 16)) {
    const int64_t nvec = n * es / 16;
    if (nvec > 0) {
      int64_t grid = (nvec + kAmaxThreads * U - 1) / (kAmaxThreads * U);
      if (grid > kAmaxBlocks) grid = kAmaxBlocks;
      if (x_dtype == MI355Q_BF16) amax_vec<true, U><<<(unsigned)grid, kAmaxThreads, 0, st>>>(xb, nvec, am);
      else amax_vec<false, U><<<(unsigned)grid, kAmaxThreads, 0, st>>>(xb, nvec, am);
      done = nvec * (16 / es);
    }
  }
  if (done < n) {
    const int64_t grid = (n - done + kThreads - 1) / kThreads;
    if (grid > 0x7fffffffLL) return MI355Q_ERR_UNSUPPORTED;
    if (x_dtype == MI355Q_BF16) amax_generic<true><<<(unsigned)grid, kThreads, 0, st>>>(xb, done, n, am);
    else amax_generic<false><<<(unsigned)grid, kThreads, 0, st>>>(xb, done, n, am);
  }
  return launch_status();
}

int mi355q_rowwise_amax(const void* x, int x_dtype, int64_t rows, int64_t cols, float* amax_out,
                        void* stream) {
  if (rows < 0 || cols < 0) return MI355Q_ERR_INVALID_ARGUMENT;
  if (rows == 0) return MI355Q_OK;
  if (amax_out == nullptr || (cols > 0 && x == nullptr)) return MI355Q_ERR_INVALID_ARGUMENT;
  if (x_dtype != MI355Q_F32 && x_dtype != MI355Q_BF16) return MI355Q_ERR_INVALID_ARGUMENT;
  if (rows > 0x7fffffffLL) return MI355Q_ERR_UNSUPPORTED;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int es = x_dtype == MI355Q_BF16 ? 2 : 4;
  const int vec_ok = aligned(x, 16) && (cols * es) % 16 == 0;
  const uint8_t* xb = static_cast<const uint8_t*>(x);
  if (x_dtype == MI355Q_BF16) rowwise_amax_kernel<true><<<(unsigned)rows, kThreads, 0, st>>>(xb, cols, vec_ok, amax_out);
  else rowwise_amax_kernel<false><<<(unsigned)rows, kThreads, 0, st>>>(xb, cols, vec_ok, amax_out);
  return launch_status();
}

int mi355q_cast_to_fp8_sr(const void* x, int x_dtype, void* y, int fp8_fmt, const float* scale_dev,
                          float scale_host, int scale_mode, int64_t outer, int64_t mid, int64_t inner,
                          float* amax_out, uint64_t seed, uint64_t offset, int flush_subnormals, void* stream) {
  if (fp8_fmt != MI355Q_E4M3FN && fp8_fmt != MI355Q_E5M2) return MI355Q_ERR_INVALID_ARGUMENT;
  if (x_dtype != MI355Q_F32 && x_dtype != MI355Q_BF16) return MI355Q_ERR_INVALID_ARGUMENT;
  if (!scale_args_ok(scale_dev, scale_mode, outer, mid, inner)) return MI355Q_ERR_INVALID_ARGUMENT;
  const int64_t n = outer * mid * inner;
  if (n > 0 && (x == nullptr || y == nullptr)) return MI355Q_ERR_INVALID_ARGUMENT;
  hipStream_t st = static_cast<hipStream_t>(stream);
  uint32_t* am = reinterpret_cast<uint32_t*>(amax_out);
  if (am) fill_u32_kernel<<<1, 1, 0, st>>>(am, 0u);
  if (n == 0) return launch_status();
  const int64_t grid = ((n + 3) / 4 + kThreads - 1) / kThreads;
  if (grid > 0x7fffffffLL) return MI355Q_ERR_UNSUPPORTED;
  const uint8_t* xb = static_cast<const uint8_t*>(x);
  uint8_t* yb = static_cast<uint8_t*>(y);
  const unsigned g = (unsigned)grid;
  if (x_dtype == MI355Q_BF16) {
    if (fp8_fmt == MI355Q_E4M3FN) cast_to_fp8_sr_kernel<true, MI355Q_E4M3FN><<<g, kThreads, 0, st>>>(xb, yb, scale_dev, scale_host, scale_mode, n, mid, inner, seed, offset, flush_subnormals, am);
    else cast_to_fp8_sr_kernel<true, MI355Q_E5M2><<<g, kThreads, 0, st>>>(xb, yb, scale_dev, scale_host, scale_mode, n, mid, inner, seed, offset, flush_subnormals, am);
  } else {
    if (fp8_fmt == MI355Q_E4M3FN) cast_to_fp8_sr_kernel<false, MI355Q_E4M3FN><<<g, kThreads, 0, st>>>(xb, yb, scale_dev, scale_host, scale_mode, n, mid, inner, seed, offset, flush_subnormals, am);
    else cast_to_fp8_sr_kernel<false, MI355Q_E5M2><<<g, kThreads, 0, st>>>(xb, yb, scale_dev, scale_host, scale_mode, n, mid, inner, seed, offset, flush_subnormals, am);
  }
  return launch_status();
}

int mi355q_cast_to_fp8_hybrid(const void* x, int x_dtype, int64_t n, void* y_e5m2, void* y_e4m3fn,
                              const float* scale_e5m2, const float* scale_e4m3fn, int stochastic,
                              uint64_t seed, uint64_t offset, float* amax_out, void* stream) {
  if (n < 0 || (x_dtype != MI355Q_F32 && x_dtype != MI355Q_BF16)) return MI355Q_ERR_INVALID_ARGUMENT;
  if (n > 0 && (x == nullptr || y_e5m2 == nullptr || y_e4m3fn == nullptr)) return MI355Q_ERR_INVALID_ARGUMENT;
  hipStream_t st = static_cast<hipStream_t>(stream);
  uint32_t* am = reinterpret_cast<uint32_t*>(amax_out);
  if (am) fill_u32_kernel<<<1, 1, 0, st>>>(am, 0u);
  if (n == 0) return launch_status();
  const uint8_t* xb = static_cast<const uint8_t*>(x);
  uint8_t* y5 = static_cast<uint8_t*>(y_e5m2);
  uint8_t* y4 = static_cast<uint8_t*>(y_e4m3fn);
  const int64_t max_blocks = am ? kAmaxBlocks : 4 * kAmaxBlocks;
  auto grid_for = [&](int64_t steps) {
    const int64_t b = (steps + kAmaxThreads - 1) / kAmaxThreads;
    return (unsigned)(b < max_blocks ? b : max_blocks);
  };
  int64_t done = 0;
  if (aligned(x, 16) && aligned(y5, 8) && aligned(y4, 8) && n >= 8) {
    const int64_t nv = n / 8;
    if (x_dtype == MI355Q_BF16) cast_to_fp8_hybrid_kernel<true, 8><<<grid_for(nv), kAmaxThreads, 0, st>>>(xb, y5, y4, scale_e5m2, scale_e4m3fn, 0, nv * 8, stochastic, seed, offset, am);
    else cast_to_fp8_hybrid_kernel<false, 8><<<grid_for(nv), kAmaxThreads, 0, st>>>(xb, y5, y4, scale_e5m2, scale_e4m3fn, 0, nv * 8, stochastic, seed, offset, am);
    done = nv * 8;
  }
  if (done < n) {
    const int64_t rest = n - done;
    if (x_dtype == MI355Q_BF16) cast_to_fp8_hybrid_kernel<true, 1><<<grid_for(rest), kAmaxThreads, 0, st>>>(xb, y5, y4, scale_e5m2, scale_e4m3fn, done, rest, stochastic, seed, offset, am);
    else cast_to_fp8_hybrid_kernel<false, 1><<<grid_for(rest), kAmaxThreads, 0, st>>>(xb, y5, y4, scale_e5m2, scale_e4m3fn, done, rest, stochastic, seed, offset, am);
  }
  return launch_status();
}

int mi355q_split_rows_fp8x2(const void* x, int x_dtype, int64_t ldx, int64_t rows, int64_t cols, void* hi, void* lo,
                            int64_t ld, float* scale_inv, void* stream) {
  if (x_dtype != MI355Q_BF16) return MI355Q_ERR_INVALID_ARGUMENT;
  if (rows < 0 || cols < 0 || ldx < cols || ld < cols) return MI355Q_ERR_INVALID_ARGUMENT;
  if (rows == 0) return MI355Q_OK;
  if (x == nullptr || hi == nullptr || lo == nullptr || scale_inv == nullptr) return MI355Q_ERR_INVALID_ARGUMENT;
  if (ld % 16 != 0 || !aligned(hi, 16) || !aligned(lo, 16) || rows > 0x7fffffffLL) return MI355Q_ERR_UNSUPPORTED;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const uint16_t* xs = static_cast<const uint16_t*>(x);
  uint8_t* h8 = static_cast<uint8_t*>(hi);
  uint8_t* l8 = static_cast<uint8_t*>(lo);
  const unsigned grid = (unsigned)rows;
  const int64_t vpr = ld / 8;  // output vectors of a row
  if (cols % 8 == 0 && ldx % 8 == 0 && aligned(x, 16) && vpr <= 8 * kThreads) {
    if (vpr <= kThreads) split_rows_vec_kernel<1><<<grid, kThreads, 0, st>>>(xs, ldx, cols, h8, l8, ld, scale_inv);
    else if (vpr <= 2 * kThreads) split_rows_vec_kernel<2><<<grid, kThreads, 0, st>>>(xs, ldx, cols, h8, l8, ld, scale_inv);
    else if (vpr <= 4 * kThreads) split_rows_vec_kernel<4><<<grid, kThreads, 0, st>>>(xs, ldx, cols, h8, l8, ld, scale_inv);
    else split_rows_vec_kernel<8><<<grid, kThreads, 0, st>>>(xs, ldx, cols, h8, l8, ld, scale_inv);
  } else {
    split_rows_kernel<<<grid, kThreads, 0, st>>>(xs, ldx, cols, h8, l8, ld, scale_inv);
  }
  return launch_status();
}

int mi355q_quantize_rows(const void* x, int x_dtype, int64_t rows, int64_t cols, void* y, int fp8_fmt,
                         float target, float* scale_out, float* scale_inv_out, void* stream) {
  if (rows < 0 || cols < 0) return MI355Q_ERR_INVALID_ARGUMENT;
  if (fp8_fmt != MI355Q_E4M3FN && fp8_fmt != MI355Q_E5M2) return MI355Q_ERR_INVALID_ARGUMENT;
  if (x_dtype != MI355Q_F32 && x_dtype != MI355Q_BF16) return MI355Q_ERR_INVALID_ARGUMENT;
  if (rows == 0 || cols == 0) return MI355Q_OK;
  if (x == nullptr || y == nullptr) return MI355Q_ERR_INVALID_ARGUMENT;
  if (rows > 0x7fffffffLL) return MI355Q_ERR_UNSUPPORTED;
  const int epv = x_dtype == MI355Q_BF16 ? 8 : 4;
  const int64_t vpr = (cols + epv - 1) / epv;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const uint8_t* xb = static_cast<const uint8_t*>(x);
  uint8_t* yb = static_cast<uint8_t*>(y);
  if (cols % epv != 0 || !aligned(x, 16) || !aligned(y, epv)) {
    if (vpr > kMaxRaggedVectors || !aligned(x, epv == 8 ? 2 : 4)) return MI355Q_ERR_UNSUPPORTED;
    const unsigned grid = (unsigned)rows, threads = (unsigned)(((vpr + 1) / 2 + 63) / 64 * 64);
    if (x_dtype == MI355Q_BF16) {
      if (fp8_fmt == MI355Q_E4M3FN) quantize_ragged_rows_kernel<true, MI355Q_E4M3FN><<<grid, threads, 0, st>>>(xb, yb, (int)cols, target, scale_out, scale_inv_out);
      else quantize_ragged_rows_kernel<true, MI355Q_E5M2><<<grid, threads, 0, st>>>(xb, yb, (int)cols, target, scale_out, scale_inv_out);
    } else {
      if (fp8_fmt == MI355Q_E4M3FN) quantize_ragged_rows_kernel<false, MI355Q_E4M3FN><<<grid, threads, 0, st>>>(xb, yb, (int)cols, target, scale_out, scale_inv_out);
      else quantize_ragged_rows_kernel<false, MI355Q_E5M2><<<grid, threads, 0, st>>>(xb, yb, (int)cols, target, scale_out, scale_inv_out);
    }
    return launch_status();
  }
  if (x_dtype == MI355Q_BF16) {
    if (fp8_fmt == MI355Q_E4M3FN) return quantize_rows_launch<true, MI355Q_E4M3FN>(xb, yb, rows, vpr, target, scale_out, scale_inv_out, st);
    return quantize_rows_launch<true, MI355Q_E5M2>(xb, yb, rows, vpr, target, scale_out, scale_inv_out, st);
  }
  if (fp8_fmt == MI355Q_E4M3FN) return quantize_rows_launch<false, MI355Q_E4M3FN>(xb, yb, rows, vpr, target, scale_out, scale_inv_out, st);
  return quantize_rows_launch<false, MI355Q_E5M2>(xb, yb, rows, vpr, target, scale_out, scale_inv_out, st);
}

int mi355q_silu_mul_quantize_rows(const void* gate, int64_t ld_gate, const void* up, int64_t ld_up,
                                  int64_t rows, int64_t cols, void* y, int fp8_fmt, float target,
                                  void* h_out, float* scale_out, float* scale_inv_out, void* stream) {
  if (rows < 0 || cols < 0 || ld_gate < cols || ld_up < cols) return MI355Q_ERR_INVALID_ARGUMENT;
  if (fp8_fmt != MI355Q_E4M3FN && fp8_fmt != MI355Q_E5M2) return MI355Q_ERR_INVALID_ARGUMENT;
  if (rows == 0 || cols == 0) return MI355Q_OK;
  if (gate == nullptr || up == nullptr || y == nullptr) return MI355Q_ERR_INVALID_ARGUMENT;
  if (rows > 0x7fffffffLL) return MI355Q_ERR_UNSUPPORTED;
  // whole 16-byte vectors only; the row has to fit the registers of one workgroup
  if (cols % 8 != 0 || ld_gate % 8 != 0 || ld_up % 8 != 0 || !aligned(gate, 16) || !aligned(up, 16) ||
      !aligned(y, 8) || (h_out && !aligned(h_out, 16)))
    return MI355Q_ERR_UNSUPPORTED;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const uint16_t* g = static_cast<const uint16_t*>(gate);
  const uint16_t* u = static_cast<const uint16_t*>(up);
  uint8_t* yb = static_cast<uint8_t*>(y);
  uint16_t* hb = static_cast<uint16_t*>(h_out);
  if (fp8_fmt == MI355Q_E4M3FN)
    return silu_mul_quantize_rows_launch<MI355Q_E4M3FN>(g, ld_gate, u, ld_up, yb, hb, rows, cols / 8, target, scale_out, scale_inv_out, st);
  return silu_mul_quantize_rows_launch<MI355Q_E5M2>(g, ld_gate, u, ld_up, yb, hb, rows, cols / 8, target, scale_out, scale_inv_out, st);
}

static int cast_to_fp8_rne(const void* x, int x_dtype, void* y, int fp8_fmt, const float* scale_dev,
                       float scale_host, int scale_mode, int64_t outer, int64_t mid, int64_t inner,
                       float* amax_out, bool zero_amax, float* next_amax, void* stream) {
  if (fp8_fmt != MI355Q_E4M3FN && fp8_fmt != MI355Q_E5M2) return MI355Q_ERR_INVALID_ARGUMENT;
  if (!scale_args_ok(scale_dev, scale_mode, outer, mid, inner)) return MI355Q_ERR_INVALID_ARGUMENT;
  const int64_t n = outer * mid * inner;
  if (n > 0 && (x == nullptr || y == nullptr)) return MI355Q_ERR_INVALID_ARGUMENT;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const uint8_t* xb = static_cast<const uint8_t*>(x);
  uint8_t* yb = static_cast<uint8_t*>(y);

  if (x_dtype == MI355Q_E4M3FN || x_dtype == MI355Q_E5M2) {
    // fp8 in, same fp8 out: identity copy, no amax (fp8_ops.cpp:201-215)
    if (x_dtype != fp8_fmt || amax_out != nullptr) return MI355Q_ERR_INVALID_ARGUMENT;
    if (n == 0) return MI355Q_OK;
    int64_t done = 0;
    if (aligned(x, 16) && aligned(y, 16) && n >= 16) {
      const int64_t nvec = n / 16;
      if ((nvec + kThreads * kCopyU - 1) / (kThreads * kCopyU) > 0x7fffffffLL) return MI355Q_ERR_UNSUPPORTED;
      copy_vec16_kernel<<<blocks_for(nvec, kThreads * kCopyU), kThreads, 0, st>>>(xb, yb, nvec);
      done = nvec * 16;
    }
    if (done < n)
      copy_bytes_kernel<<<blocks_for(n - done, kThreads), kThreads, 0, st>>>(xb + done, yb + done, n - done);
    return launch_status();
  }
  if (x_dtype != MI355Q_F32 && x_dtype != MI355Q_BF16) return MI355Q_ERR_INVALID_ARGUMENT;

  uint32_t *am = reinterpret_cast<uint32_t*>(amax_out), *next = reinterpret_cast<uint32_t*>(next_amax);
  if (am && zero_amax) fill_u32_kernel<<<1, 1, 0, st>>>(am, 0u);
  if (n == 0) {
    if (next) fill_u32_kernel<<<1, 1, 0, st>>>(next, 0u);
    return launch_status();
  }
  if (x_dtype == MI355Q_BF16) {
    if (fp8_fmt == MI355Q_E4M3FN) return cast_to_dispatch<true, MI355Q_E4M3FN>(xb, yb, scale_dev, scale_host, scale_mode, outer, mid, inner, am, next, st);
    return cast_to_dispatch<true, MI355Q_E5M2>(xb, yb, scale_dev, scale_host, scale_mode, outer, mid, inner, am, next, st);
  }
  if (fp8_fmt == MI355Q_E4M3FN) return cast_to_dispatch<false, MI355Q_E4M3FN>(xb, yb, scale_dev, scale_host, scale_mode, outer, mid, inner, am, next, st);
  return cast_to_dispatch<false, MI355Q_E5M2>(xb, yb, scale_dev, scale_host, scale_mode, outer, mid, inner, am, next, st);
}

int mi355q_cast_to_fp8(const void* x, int x_dtype, void* y, int fp8_fmt, const float* scale_dev,
                       float scale_host, int scale_mode, int64_t outer, int64_t mid, int64_t inner,
                       float* amax_out, void* stream) {
  return cast_to_fp8_rne(x, x_dtype, y, fp8_fmt, scale_dev, scale_host, scale_mode, outer, mid, inner, amax_out, true, nullptr, stream);
}

int mi355q_cast_to_fp8_running_amax(const void* x, int x_dtype, void* y, int fp8_fmt, const float* scale_dev,
                                    float scale_host, int scale_mode, int64_t outer, int64_t mid, int64_t inner,
                                    float* running_amax, void* stream) {
  if (running_amax == nullptr) return MI355Q_ERR_INVALID_ARGUMENT;
  return cast_to_fp8_rne(x, x_dtype, y, fp8_fmt, scale_dev, scale_host, scale_mode, outer, mid, inner, running_amax, false, nullptr, stream);
}

int mi355q_cast_to_fp8_amax_chain(const void* x, int x_dtype, void* y, int fp8_fmt, const float* scale_dev,
                                  float scale_host, int scale_mode, int64_t outer, int64_t mid, int64_t inner,
                                  float* amax, int amax_is_zero, float* next_amax, void* stream) {
  if (amax == nullptr || amax == next_amax) return MI355Q_ERR_INVALID_ARGUMENT;
  return cast_to_fp8_rne(x, x_dtype, y, fp8_fmt, scale_dev, scale_host, scale_mode, outer, mid, inner, amax, amax_is_zero == 0, next_amax, stream);
}

int mi355q_cast_from_fp8(const void* x, int fp8_fmt, void* y, int out_dtype, const float* scale_dev,
                         float scale_host, int scale_mode, int64_t outer, int64_t mid,
                         int64_t inner, void* stream) {
  if (fp8_fmt != MI355Q_E4M3FN && fp8_fmt != MI355Q_E5M2) return MI355Q_ERR_INVALID_ARGUMENT;
  if (out_dtype != MI355Q_F32 && out_dtype != MI355Q_BF16) return MI355Q_ERR_INVALID_ARGUMENT;
  if (!scale_args_ok(scale_dev, scale_mode, outer, mid, inner)) return MI355Q_ERR_INVALID_ARGUMENT;
  const int64_t n = outer * mid * inner;
  if (n == 0) return MI355Q_OK;
  if (x == nullptr || y == nullptr) return MI355Q_ERR_INVALID_ARGUMENT;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const uint8_t* xb = static_cast<const uint8_t*>(x);
  uint8_t* yb = static_cast<uint8_t*>(y);
  if (fp8_fmt == MI355Q_E4M3FN) {
    if (out_dtype == MI355Q_BF16) return cast_from_dispatch<MI355Q_E4M3FN, true>(xb, yb, scale_dev, scale_host, scale_mode, outer, mid, inner, st);
    return cast_from_dispatch<MI355Q_E4M3FN, false>(xb, yb, scale_dev, scale_host, scale_mode, outer, mid, inner, st);
  }
  if (out_dtype == MI355Q_BF16) return cast_from_dispatch<MI355Q_E5M2, true>(xb, yb, scale_dev, scale_host, scale_mode, outer, mid, inner, st);
  return cast_from_dispatch<MI355Q_E5M2, false>(xb, yb, scale_dev, scale_host, scale_mode, outer, mid, inner, st);
}

int mi355q_pad_rows(const mi355q_pad_desc* desc, int count, void* stream) {
  if (desc == nullptr || count < 1 || count > 2) return MI355Q_ERR_INVALID_ARGUMENT;
  PadJobs jobs{};
  int64_t blocks[2] = {0, 0};
  for (int i = 0; i < count; ++i) {
    const mi355q_pad_desc& d = desc[i];
    if (d.batch < 0 || d.rows < 0 || d.cols < 0 || d.dst_rows < d.rows || d.dst_ld < d.cols || d.dst_ld % 16 || d.src_ld < d.cols)
      return MI355Q_ERR_INVALID_ARGUMENT;
    if (d.batch == 0 || d.dst_rows == 0 || d.dst_ld == 0) continue;
    if (d.dst == nullptr || !aligned(d.dst, 16) || (d.rows > 0 && d.cols > 0 && d.src == nullptr)) return MI355Q_ERR_INVALID_ARGUMENT;
    if (d.rows > 0x7fffffffLL || d.dst_rows > 0x7fffffffLL || d.dst_ld > 0x7fffffffLL || d.batch > 0x7fffffffLL) return MI355Q_ERR_UNSUPPORTED;
    PadJob& j = jobs.job[i];
    j.src = static_cast<const uint8_t*>(d.src);
    j.dst = static_cast<uint8_t*>(d.dst);
    j.src_ld = d.src_ld;
    j.src_stride = d.src_stride;
    j.dst_stride = d.dst_rows * d.dst_ld;
    j.rows = (int32_t)d.rows;
    j.cols = (int32_t)d.cols;
    j.dst_rows = (int32_t)d.dst_rows;
    j.dst_chunks = (int32_t)(d.dst_ld / 16);
    j.batch = (int32_t)d.batch;
    j.chunks = d.batch * d.dst_rows * (d.dst_ld / 16);
    blocks[i] = (j.chunks + kThreads * kPadU - 1) / (kThreads * kPadU);
  }
  if (blocks[0] + blocks[1] == 0) return MI355Q_OK;
  if (blocks[0] + blocks[1] > 0x7fffffffLL) return MI355Q_ERR_UNSUPPORTED;
  pad_rows_kernel<<<(unsigned)(blocks[0] + blocks[1]), kThreads, 0, static_cast<hipStream_t>(stream)>>>(jobs, blocks[0]);
  return launch_status();
}

}  // extern "C"
