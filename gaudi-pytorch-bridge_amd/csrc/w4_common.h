// What the kernels of w4_gemm.hip and w4_stream.h share: their arguments, the global -> LDS load of one piece per lane, and the
// epilogue of four columns of a row.
#pragma once
#include "gemm_tile.h"

namespace mi355q {

constexpr size_t kW4TicketBytes = 1024;  // the counters in front of a workspace, the same for every shape

struct W4Args {
  GemmArgs g;              // A, C, M, N, K, lda, ldc, sa*, bias*, out_bf16 (B, sb*, D unused)
  const uint8_t* packed;   // int32 [K, N / 8]
  int64_t ld_packed;       // bytes between k-rows
  const uint8_t* scale;    // [K / group, N] bf16 or fp32
  const uint8_t* zp;       // packed int32 [K / group, N / 8] or nullptr
  int scale_f32, is_signed;
  int stages_per_group;    // group / 128
  // wide and stream kernels: K is walked in `ksplit` parts by as many workgroups per strip
  int ksplit;
  uint32_t* tickets;       // one per strip, zero between launches
  float* partials;         // partial sums [ksplit][strips], in the consumers' register order: the wide kernel's tiles of its rows x 256, the stream kernel's 16 x 512
  int ticket_stride;       // stream kernel: 32-bit words between the counters
  // 16-bit activations as two fp8 planes (wide kernel, A16): g.A holds the leading part of every value and a_lo,
  // with the same pitch, 16 times what is left of it (split_rows_kernel); a = (A + a_lo / 16) / row scale
  const uint8_t* a_lo;
};

// One 16-byte piece per lane, straight copy into LDS (lane l lands at dst + 16 l).  The
// s_nop covers a descriptor word that reached its scalar register through a vector
// instruction (five wait states before a memory instruction may read it).
// STREAM adds the nontemporal hint, for weights that the launch reads once.
template <bool STREAM = false>
__device__ __forceinline__ void w4_dma16(const i32x4& rsrc, int voff, uint32_t lds_dst) {
  if constexpr (STREAM) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tbuffer_load_dwordx4 %1, %2, 0 offen nt lds"
                 :
                 : "s"(lds_dst), "v"(voff), "s"(rsrc)
                 : "memory", "m0");
  } else {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                 :
                 : "s"(lds_dst), "v"(voff), "s"(rsrc)
                 : "memory", "m0");
  }
}

// The same with four bytes per lane (lane l lands at dst + 4 l).
__device__ __forceinline__ void w4_dma4(const i32x4& rsrc, int voff, uint32_t lds_dst) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tbuffer_load_dword %1, %2, 0 offen lds" : : "s"(lds_dst), "v"(voff), "s"(rsrc) : "memory", "m0");
}

// The row that lane i of a group of 16 addresses in a transposing LDS read for nibbles that end up as bytes (w4_bytes in w4_gemm.hip).
__device__ __forceinline__ int w4_nibble_row(int i) { return (i & 8) | ((i & 1) << 2) | ((i >> 1) & 3); }

// What the epilogue multiplies a row by and adds to its columns.  Loaded for all of a lane's results before the first is stored: a
// load behind a store waits for a trip to the L2 of its own, and a lane of a 128-row tile has
// sixteen (uint4, us, before and after: 512 x 4096 x 16384 54.5 -> 51.8, two planes 74.5 -> 70.9; 60 x 4096 x 40960 36.3 -> 34.7,
// 41.7 -> 40.5; 133 x 10112 x 21696 two planes 140.5 -> 135.5; parts added up by a second launch +- 0).  (Rows and columns past the
// edge read the last ones; they are not stored.)
__device__ __forceinline__ float w4_row_scale(const GemmArgs& g, const ScalarScales& scalars, int m) {
  return g.sa_mode == MI355Q_GS_PER_ROW ? g.sa[m < g.M ? m : g.M - 1] : scalars.sa;
}
__device__ __forceinline__ f32x4 w4_bias4(const GemmArgs& g, int n) {
  f32x4 b = {0.f, 0.f, 0.f, 0.f};
  if (g.bias_mode == MI355Q_BIAS_ROW_VECTOR) {
    const int from = n < g.N ? n : g.N - 4;
#pragma unroll
    for (int e = 0; e < 4; ++e) b[e] = load_out_as_f32(g.bias, from + e, g.out_bf16);
  }
  return b;
}

// The epilogue of four columns of a row: N is a multiple of 32, so they are inside or outside together.
__device__ __forceinline__ void w4_store4(const GemmArgs& g, int m, int n, const f32x4& sums, float sa, const f32x4& bias) {
  if (m >= g.M || n >= g.N) return;
  const int es = g.out_bf16 ? 2 : 4;
  float v[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = __fmul_rn(sums[e], sa) + bias[e];  // rounded as the other epilogues round
  uint8_t* cp = g.C + ((int64_t)m * g.ldc + n) * es;
  const bool vec_ok = (reinterpret_cast<uintptr_t>(cp) % (4 * es)) == 0;
  if (g.out_bf16) {
    if (vec_ok) {
      *reinterpret_cast<u32x2*>(cp) = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) reinterpret_cast<uint16_t*>(cp)[e] = (uint16_t)(pack_bf16x2(v[e], v[e]) & 0xffffu);
    }
  } else {
    if (vec_ok) {
      *reinterpret_cast<f32x4*>(cp) = f32x4{v[0], v[1], v[2], v[3]};
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) reinterpret_cast<float*>(cp)[e] = v[e];
    }
  }
}

}  // namespace mi355q
