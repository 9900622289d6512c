// fp8 GEMM for at most 16 rows of A, K-major, against B [K, N] (decode-shaped calls in the usual weight layout).
//
// Such a product is bound by reading B once.  B goes from memory straight into vector registers: no LDS, no
// barrier and no descriptor arithmetic stand between a wave and its next load, every wave streams on its own, and
// 256 KiB (8 waves of 32 KiB) are on their way into a compute unit all the time.  A workgroup of eight waves owns 256
// columns of C and one part of K; its waves take 32 k of that part in turns, add their sums up through LDS at the
// end, and the workgroups that share columns meet through the workspace (gemm_split.h).
//
// A k-row of the strip is 256 bytes: lane i of a 16-lane group loads 16 neighbouring columns of it and a group takes
// 8 consecutive k-rows, so that a load instruction covers whole rows of the strip.  The 8 x 16 bytes a lane then holds
// are transposed in registers (v_perm_b32, four k by four columns at a time), and column t of every lane is one
// operand of v_mfma_f32_16x16x32: MFMA t multiplies the columns { 16 lane + t }.  The transposition takes 64 v_perm
// per 8 KiB and wave, a tenth of the stream's time, under which it hides.
//
// Strips of 256 columns because 256-byte pieces of such a matrix stream at 6.65 TB/s and 128-byte ones at 5.8 (strip
// reads alone, 235 MB: 35.3 against 40.3 us); with 8-byte loads (strips of 128 columns here) it was 5.0.  Measured at
// 16 x 8192 x 28672: 38.9 us for the stream, 1.8 for the sum over the waves and the epilogue, 2.2 for the meeting of
// the two parts of K: 43 us (ring kernel of gemm_ring.h: 46.4).  Below about 100 MB of B the ring kernel's shorter start
// and end win (16 x 8192 x 8192: 18.9 against 15.1 us).  A second row tile (M <= 32) leaves room for half the loads in flight
// and loses as well (48 against 46.5 us), and so does a K-major B, loaded in 64-byte pieces per row (52 against 40).
#pragma once
#include "gemm_split.h"

namespace mi355q {

constexpr int kStWaves = 8;
constexpr int kStThreads = kStWaves * 64;
constexpr int kStRows = 16;
constexpr int kStBN = 256;

struct StreamArgs {
  GemmArgs g;
  int strips;          // ceil(N / kStBN)
  SplitArgs split;     // a counter and `parts` tiles of sums for each of the batch * strips strips
};

template <int FMT_B, int FMT_A>
__device__ __forceinline__ f32x4 st_mfma32(u32x2 b, u32x2 a, f32x4 c) {
  const long bl = __builtin_bit_cast(long, b), al = __builtin_bit_cast(long, a);
  if constexpr (FMT_B == MI355Q_E4M3FN && FMT_A == MI355Q_E4M3FN) return __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(bl, al, c, 0, 0, 0);
  else if constexpr (FMT_B == MI355Q_E4M3FN) return __builtin_amdgcn_mfma_f32_16x16x32_fp8_bf8(bl, al, c, 0, 0, 0);
  else if constexpr (FMT_A == MI355Q_E4M3FN) return __builtin_amdgcn_mfma_f32_16x16x32_bf8_fp8(bl, al, c, 0, 0, 0);
  else return __builtin_amdgcn_mfma_f32_16x16x32_bf8_bf8(bl, al, c, 0, 0, 0);
}

// bytes b of w0 .. w3 (four k of four columns) -> four words, word j = column j's four k
__device__ __forceinline__ void st_transpose4(uint32_t w0, uint32_t w1, uint32_t w2, uint32_t w3, uint32_t (&o)[4]) {
  const uint32_t t0 = __builtin_amdgcn_perm(w1, w0, 0x05010400u), t1 = __builtin_amdgcn_perm(w1, w0, 0x07030602u);
  const uint32_t u0 = __builtin_amdgcn_perm(w3, w2, 0x05010400u), u1 = __builtin_amdgcn_perm(w3, w2, 0x07030602u);
  o[0] = __builtin_amdgcn_perm(u0, t0, 0x05040100u);
  o[1] = __builtin_amdgcn_perm(u0, t0, 0x07060302u);
  o[2] = __builtin_amdgcn_perm(u1, t1, 0x05040100u);
  o[3] = __builtin_amdgcn_perm(u1, t1, 0x07060302u);
}

// Row and column factors and the bias vector of the workgroup's rows and columns, fetched before the stream starts
// (read at its end they would be cold misses, one after the other, with nothing left to hide them under).  A's scale and
// B's stay apart, one as the row's factor and one as the column's: their product can leave fp32's range where neither
// sums nor results do.  Where both are per row, or both per column, the second one is B's.
struct StreamFactors {
  float row[kStRows], col[kStBN], bias[kStBN], second[kStBN];
};
__device__ __forceinline__ bool st_two_of_a_kind(const GemmArgs& g) {
  return g.sa_mode == g.sb_mode && (g.sa_mode == MI355Q_GS_PER_ROW || g.sa_mode == MI355Q_GS_PER_COL);
}
// Requested without a branch (a factor the problem does not have is an empty buffer, which reads as zero and touches
// no memory): a branch here would make the compiler wait for the values in front of the stream's first loads.
struct StreamFactorLoads {
  uint32_t a_col, b_col, a_row, b_row, bias32;
  uint16_t bias16;
  __device__ __forceinline__ static uint32_t word(const void* p, int count, int i) {
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, count * 4, 0x00020000);
    return __builtin_amdgcn_raw_buffer_load_b32(r, i * 4, 0, 0);
  }
  __device__ __forceinline__ void request(const GemmArgs& g, int64_t batch, int n0) {
    const int n = n0 + (int)threadIdx.x, m = threadIdx.x;
    const auto rows = [&](int mode) { return mode == MI355Q_GS_PER_ROW ? g.M : (mode == MI355Q_GS_DEV ? 1 : 0); };
    a_col = word(g.sa, g.sa_mode == MI355Q_GS_PER_COL ? g.N : 0, n);
    b_col = word(g.sb, g.sb_mode == MI355Q_GS_PER_COL ? g.N : 0, n);
    a_row = word(g.sa, rows(g.sa_mode), g.sa_mode == MI355Q_GS_PER_ROW ? m : 0);
    b_row = word(g.sb, rows(g.sb_mode), g.sb_mode == MI355Q_GS_PER_ROW ? m : 0);
    const bool vec = g.bias_mode == MI355Q_BIAS_ROW_VECTOR;
    const uint8_t* bias = g.bias + batch * g.stride_bias * (g.out_bf16 ? 2 : 4);
    bias32 = word(bias, vec && !g.out_bf16 ? g.N : 0, n);
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(bias), 0, vec && g.out_bf16 ? g.N * 2 : 0, 0x00020000);
    bias16 = __builtin_amdgcn_raw_buffer_load_b16(r, n * 2, 0, 0);
  }
  __device__ __forceinline__ void keep(const GemmArgs& g, StreamFactors& f) const {
    const auto scalar = [&](int mode, float host, uint32_t loaded) {
      return mode == MI355Q_GS_HOST ? host : (mode == MI355Q_GS_DEV || mode == MI355Q_GS_PER_ROW ? __uint_as_float(loaded) : 1.0f);
    };
    const float a_here = scalar(g.sa_mode, g.sa_host, a_row), b_here = scalar(g.sb_mode, g.sb_host, b_row);
    const bool a_in_col = g.sa_mode == MI355Q_GS_PER_COL, b_in_col = g.sb_mode == MI355Q_GS_PER_COL;
    const bool a_in_row = g.sa_mode == MI355Q_GS_PER_ROW, b_in_row = g.sb_mode == MI355Q_GS_PER_ROW;
    // the row's factor is A's scale and the column's B's, scalars too, but where A's is per column or only B's per row
    const bool turned = (a_in_col && !b_in_col) || (b_in_row && !a_in_row);
    if (threadIdx.x < kStBN) {
      f.col[threadIdx.x] = a_in_col ? __uint_as_float(a_col) : (turned ? a_here : (b_in_col ? __uint_as_float(b_col) : b_here));
      f.bias[threadIdx.x] = g.out_bf16 ? bf16_bits_to_f32(bias16) : __uint_as_float(bias32);
      if (st_two_of_a_kind(g)) f.second[threadIdx.x] = b_in_col ? __uint_as_float(b_col) : b_here;
    }
    if (threadIdx.x < kStRows) f.row[threadIdx.x] = turned ? b_here : a_here;
  }
};

// Eight consecutive columns of one row: scales, bias and accumulate input in fp32, one rounding, stored.
__device__ __forceinline__ void st_store8(const GemmArgs& g, int64_t batch, int m, int n0, int col, const float (&acc)[8],
                                          const StreamFactors& f) {
  const int n = n0 + col;
  if (m >= g.M || n >= g.N) return;
  const int es = g.out_bf16 ? 2 : 4;
  const float rf = f.row[m];
  float v[8];
  if (st_two_of_a_kind(g)) {
    const bool rows = g.sa_mode == MI355Q_GS_PER_ROW;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = __builtin_fmaf(acc[e] * (rows ? rf : f.col[col + e]), f.second[rows ? m : col + e], f.bias[col + e]);
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = __builtin_fmaf(acc[e] * rf, f.col[col + e], f.bias[col + e]);
  }
  if (g.D != nullptr || g.bias_mode == MI355Q_BIAS_FULL) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int ne = n + e < g.N ? n + e : g.N - 1;
      if (g.bias_mode == MI355Q_BIAS_FULL) v[e] += load_out_as_f32(g.bias + batch * g.stride_bias * es, (int64_t)m * g.ldbias + ne, g.out_bf16);
      if (g.D) v[e] += load_out_as_f32(g.D + batch * g.stride_d * es, (int64_t)m * g.ldd + ne, g.out_bf16);
    }
  }
  uint8_t* cp = g.C + batch * g.stride_c * es + ((int64_t)m * g.ldc + n) * es;
  const bool vec = n + 8 <= g.N && (reinterpret_cast<uintptr_t>(cp) & 15u) == 0;
  if (g.out_bf16) {
    if (vec) {
      *reinterpret_cast<u32x4*>(cp) = u32x4{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7])};
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (n + e < g.N) reinterpret_cast<uint16_t*>(cp)[e] = (uint16_t)(pack_bf16x2(v[e], v[e]) & 0xffffu);
    }
  } else if (vec) {
    reinterpret_cast<f32x4*>(cp)[0] = f32x4{v[0], v[1], v[2], v[3]};
    reinterpret_cast<f32x4*>(cp)[1] = f32x4{v[4], v[5], v[6], v[7]};
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (n + e < g.N) reinterpret_cast<float*>(cp)[e] = v[e];
  }
}

template <int FMT_A, int FMT_B>
__global__ __launch_bounds__(kStThreads, 2) void fp8_gemm_stream_kernel(StreamArgs a) {
  constexpr int NT = kStBN / 16;                     // MFMA column tiles, and columns per lane
  constexpr int kTilesPerWave = NT / kStWaves;       // in the sum over the waves
  constexpr int kOutPitch = kStBN + 4;
  constexpr int S = 4;                               // units (of 32 k) in flight per wave
  __shared__ __attribute__((aligned(16))) f32x4 red[kStWaves][NT][64];
  __shared__ __attribute__((aligned(16))) float outs[kStRows * kOutPitch];
  __shared__ StreamFactors factors;
  __shared__ uint32_t ticket;

  const GemmArgs& g = a.g;
  const int64_t batch = blockIdx.y;
  const int strip = blockIdx.x % a.strips, part = blockIdx.x / a.strips;
  const int n0 = strip * kStBN;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, i16 = lane & 15, gk = lane >> 4;
  const int units = (g.K + 31) / 32;
  const int u0 = (int)((int64_t)part * units / a.split.parts), u1 = (int)((int64_t)(part + 1) * units / a.split.parts);
  const uint8_t* Ab = g.A + batch * g.stride_a;
  const uint8_t* Bb = g.B + batch * g.stride_b;
  constexpr int kOut = 0x7fffffff;  // an offset no descriptor reaches: reads as zero, touches no memory
  const int lda = (int)g.lda, ldb = (int)g.ldb;
  const int n16 = (g.N + 15) & ~15;                  // ldb is a multiple of 16 and at least N
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(Ab), 0, (g.M - 1) * lda + g.K, 0x00020000);
  const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(Bb + n0), 0, (g.K - 1) * ldb + (n16 - n0), 0x00020000);
  const bool col_ok = n0 + NT * i16 < n16, row_ok = i16 < g.M;

  f32x4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  StreamFactorLoads factor_loads;
  factor_loads.request(g, batch, n0);

  u32x4 buf[S][8];
  u32x2 abuf[S];
  // unit u: k-rows 32 u + 8 gk + r of B (the hint: read once) and the same k of A's row; units past the part's end and
  // k past K (K is a multiple of 16: eight rows are inside or outside together) read as zero
  auto load = [&](auto sc, int u) {
    constexpr int s = decltype(sc)::value;
    const int k = 32 * u + 8 * gk;
    const bool ok = u < u1 && k < g.K;
    const int vb = ok && col_ok ? k * ldb + NT * i16 : kOut;
#pragma unroll
    for (int r = 0; r < 8; ++r) buf[s][r] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rb, vb, r * ldb, 2));
    abuf[s] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(ra, ok && row_ok ? i16 * lda + k : kOut, 0, 0));
  };
  auto multiply = [&](auto sc) {
    constexpr int s = decltype(sc)::value;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      uint32_t lo[4], hi[4];
      st_transpose4(buf[s][0][d], buf[s][1][d], buf[s][2][d], buf[s][3][d], lo);
      st_transpose4(buf[s][4][d], buf[s][5][d], buf[s][6][d], buf[s][7][d], hi);
#pragma unroll
      for (int b = 0; b < 4; ++b) acc[4 * d + b] = st_mfma32<FMT_B, FMT_A>(u32x2{lo[b], hi[b]}, abuf[s], acc[4 * d + b]);
    }
  };
  int u = u0 + wave;
  static_for<S>([&](auto sc) { load(sc, u + kStWaves * decltype(sc)::value); });
  factor_loads.keep(g, factors);
  for (; u < u1; u += kStWaves * S) {
    static_for<S>([&](auto sc) {
      multiply(sc);
      __builtin_amdgcn_sched_barrier(0);
      load(sc, u + kStWaves * (S + decltype(sc)::value));
      __builtin_amdgcn_sched_barrier(0);
    });
  }

  // the eight waves' sums: lane (m = lane % 16, gk) of tile t holds columns 16 (4 gk + e) + t of the strip
  const int slots = a.strips * gridDim.y, slot = (int)batch * a.strips + strip;
  if (a.split.parts > 1 && threadIdx.x == 0) ticket = split_look(a.split, slot);
#pragma unroll
  for (int t = 0; t < NT; ++t) red[wave][t][lane] = acc[t];
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kTilesPerWave; ++j) {
    const int t = wave * kTilesPerWave + j;
    f32x4 s = red[0][t][lane];
#pragma unroll
    for (int w = 1; w < kStWaves; ++w) {
      const f32x4 v = red[w][t][lane];
#pragma unroll
      for (int e = 0; e < 4; ++e) s[e] += v[e];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) outs[i16 * kOutPitch + NT * (4 * gk + e) + t] = s[e];
  }
  __syncthreads();
  // a thread takes eight columns of one row
  const int row = threadIdx.x / (kStBN / 8), col = (threadIdx.x % (kStBN / 8)) * 8;
  static_assert(kStThreads == kStRows * (kStBN / 8), "one row of eight columns per thread");
  float vals[8];
  const f32x4 lo = *reinterpret_cast<const f32x4*>(outs + row * kOutPitch + col), hi = *reinterpret_cast<const f32x4*>(outs + row * kOutPitch + col + 4);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    vals[e] = lo[e];
    vals[4 + e] = hi[e];
  }
  if (a.split.parts > 1) {
    const bool others_in = ticket == (uint32_t)a.split.parts - 1;
    __syncthreads();
    if (!split_exchange<8, kStThreads>(a.split, slot, slots, part, row < g.M, others_in, &ticket, [&](int j) { return vals[j]; },
                                       [&](int j, float v) { vals[j] = v; }))
      return;
  }
  st_store8(g, batch, row, n0, col, vals, factors);
}

template <int FA, int FB>
void launch_stream(const GemmArgs& g, const SplitPlan& p, const SplitArgs& split, int64_t batch, hipStream_t st) {
  const StreamArgs a{g, p.strips, split};
  dim3 grid((unsigned)(p.strips * split.parts), (unsigned)batch);
  fp8_gemm_stream_kernel<FA, FB><<<grid, kStThreads, 0, st>>>(a);
}

}  // namespace mi355q
