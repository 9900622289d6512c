// fp8 GEMM on tiles of 16 to 256 rows and 128 columns, for every product that does not fill the chip with 256 x 256 tiles:
// one tile per workgroup, a ring of LDS stages of 128 k, v_mfma_f32_16x16x128_f8f6f4, K whole or in parts over workgroups.
//
// What bounds it.  A compute unit keeps about 32 KB of lines on their way, whatever asks for them (a loop that only loads, into
// LDS or registers, 4 to 16 waves: 48 to 55 KB/us from HBM at 0.63 us a load, 150 to 200 KB/us from the XCD's L2): its intake is
// what a stage costs, (rows + 128) x 128 bytes, and a wave that issues loads beyond that limit stalls.  Where both kinds mix, all of it
// comes at HBM's rate: 256 x 8192 x 28672 takes 64 us for a workgroup's 3 MiB (49 KB/us) though the 2 MiB of A are found in the L2
// (252 MB read from HBM in all), so A's lines, which a wave requests in turn with B's and gets back in that order, gain nothing
// from it.  Loading waves of their own for either operand have not been tried with this ring.  Hence
//  * four waves that only load and four that only multiply, one of each per SIMD, meeting at one barrier per stage: the
//    loading waves' stalls hold up no MFMA, and the multiplying waves' loop is MFMAs, fragment reads and one addition per
//    address register;
//  * as many stages as the LDS holds (3 at 256 and 192 rows, 4, 6, 7, 7 below), counted waits, and load addresses without arithmetic;
//  * low tiles where they fill the chip better, and K in parts only then (gemm_api.hip has the figures that choose);
//  * plain loads for a B of at most 64 MiB (ring_streams_b): the nontemporal hint keeps a matrix out of the 256 MB memory-side
//    cache, from which a second call would read it.
// Measured against the strip, 128 x 128 and 256 x 128 kernels it replaces (us, weights [K, N] but where nk, three sets of them in
// turn): 256 x 8192 x 28672 88.8 -> 68.3 (nk 93.3 -> 66.5; the load stream alone takes 64), 1000 x 3008 x 5000 29.3 -> 24.3, 669 x 8704 x
// 7808 nk 54.8 -> 44.7, 64 x 14336 x 4096 25.0 -> 17.5, 83 x 6640 x 864 23.9 -> 11.0, 7 x 10816 x 704 nk 16.1 -> 9.7, 1 x 4096 x 4096
// 12.2 -> 7.8.  192 rows, for A [M, K] (a K-major tile's LDS rows are 128 bytes at any height, an MN-major one's would be no power
// of two): 24 stages of 240 tiles against 160 of 256 rows, 1000 x 3008 x 5000 32.3 -> 30.6; 267 x 4736 x 28544 on tiles of 192 rows against
// 256 x 256 60.4 -> 51.9, 268 x 5296 x 13328 40.8 -> 34.4; over 480 products of 1 to 4096 rows 26 % less time in the geometric mean warm, 23 % cold.
#pragma once
#include "gemm_split.h"
#include "gemm_tile16.h"

namespace mi355q {

constexpr int kRingBN = 128;
constexpr int kRingWaves = 4;                      // that multiply, and as many that load
constexpr int kRingThreads = 2 * kRingWaves * 64;

// Global -> LDS loader of a wave's share of one operand's stages (consecutive 1 KiB regions).  What a lane fetches does not
// change from stage to stage, so its offsets are worked out once, with everything in them that the other loaders leave to
// the descriptor or test per load: tile rows past the matrix read its last row (their products are never stored, and a
// load that goes to memory retires in issue order, which the counted waits need), columns past it and, in a ragged last
// stage, k past K read as zero through an offset that no descriptor covers.  A step along K is one 64-bit scalar addition,
// whatever the operand's size.
template <bool KMAJOR, int EXT>
struct RingLoader {
  using G = TileGeom<KMAJOR, KMAJOR ? EXT : kBK, KMAJOR ? kBK : EXT, 1>;
  static constexpr int kCPR = G::kChunksPerRow, kRowsPerRegion = 64 / kCPR;
  static constexpr int kPerWave = G::kChunks / 64 / kRingWaves;
  static_assert(kPerWave * kRingWaves * 64 == G::kChunks, "tile does not split over the waves");
  static constexpr int kNowhere = 0x7fffffff;
  uint64_t base;  // the next stage to load
  int64_t step;
  int at[kPerWave], limit[kPerWave];  // a lane's offsets in a stage, lowered by issue()'s immediate, and their k in it
  int cur[kPerWave];                  // those of the next stage's loads
  int wave;

  // p: the operand at the tile's first row (column) and the workgroup's first k; valid: rows (columns) from there to the edge
  __device__ __forceinline__ void init(const uint8_t* p, int64_t ld, int valid, int wave_) {
    wave = wave_;
    const uint64_t b = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(b >> 32));
    base = ((uint64_t)hi << 32) | lo;
    step = KMAJOR ? kBK : (int64_t)kBK * ld;
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i < kPerWave; ++i) {
      const int row = (wave * kPerWave + i) * kRowsPerRegion + lane / kCPR;
      const int c16 = ((lane % kCPR) ^ G::swizzle(row)) * 16;
      int v;
      if constexpr (KMAJOR) v = (row < valid ? row : valid - 1) * (int)ld + c16;
      else v = c16 < ((valid + 15) & ~15) ? row * (int)ld + c16 : kNowhere;  // (the chunk that straddles the edge lies in the row's padding)
      at[i] = v - (i & 3) * 1024;
      limit[i] = KMAJOR ? c16 : row;
      cur[i] = at[i];
    }
  }
  // The next stage's loads read zeros from its k `valid_k` on (kBK: all of it is inside K).
  __device__ __forceinline__ void select(int valid_k) {
#pragma unroll
    for (int i = 0; i < kPerWave; ++i) cur[i] = limit[i] < valid_k ? at[i] : kNowhere - (i & 3) * 1024;
  }
  // Load I of the next stage into the operand's tile at LDS address `tile`.  Four loads in a row share a write of m0 (see
  // DmaLoader::issue_one); NT: the operand is read once.
  template <int I, bool NT>
  __device__ __forceinline__ void issue(uint32_t tile) const {
    constexpr int r = I & 3;
    const i32x4 rsrc = {(int)(uint32_t)base, (int)((uint32_t)(base >> 32) & 0xffffu), 0x7ffffff0, 0x00020000};
    if constexpr (r == 0) {
      const uint32_t dst = tile + (uint32_t)((wave * kPerWave + I) * 1024);
      if constexpr (NT) asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen nt lds" : : "s"(dst), "v"(cur[I]), "s"(rsrc) : "memory", "m0");
      else asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" : : "s"(dst), "v"(cur[I]), "s"(rsrc) : "memory", "m0");
    } else {
      if constexpr (NT) asm volatile("buffer_load_dwordx4 %0, %1, 0 offen offset:%2 nt lds" : : "v"(cur[I]), "s"(rsrc), "n"(r * 1024) : "memory");
      else asm volatile("buffer_load_dwordx4 %0, %1, 0 offen offset:%2 lds" : : "v"(cur[I]), "s"(rsrc), "n"(r * 1024) : "memory");
    }
  }
};

// Fragment reads of FragReader16 from a ring position that is not a compile-time constant: one addition per address
// register and stage.
template <bool KMAJOR, int EXT, int TILES>
struct RingReader : FragReader16<KMAJOR, EXT, TILES> {
  using Base = FragReader16<KMAJOR, EXT, TILES>;
  __device__ __forceinline__ void move(int bytes) {
#pragma unroll
    for (int i = 0; i < Base::kRegs; ++i) this->addr[i] += (uint32_t)bytes;
  }
};

// A wave's scales and bias (ScaleStager's layout), then room for its rows: 16 MT x 16 NT results leave through LDS.
constexpr int kRingScaleBytes = kStagedBytes;

// The fast bf16 epilogue (see epilogue_fast_ok) for wave tiles of 16 MT x 16 NT: epilogue16_bf16_fast with rows of 32 NT bytes.
// Write cycles (16 rows, two neighbouring 8-byte slots) and read cycles (whole rows, 16-byte chunks) touch distinct banks.
template <int MT, int NT, bool PER_COL, bool HAS_BIAS>
__device__ __forceinline__ void ring_epilogue_fast(const GemmArgs& g, int64_t batch, f32x4 (&acc)[MT][NT], int m_wave, int n_wave,
                                                   const uint8_t* staged_p, uint8_t* rows_p, ScalarScales scalars) {
  static_assert(NT == 2 || NT == 4, "64- or 128-byte rows");
  constexpr int kRow = 32 * NT, kShift = NT == 4 ? 1 : 2, kMask = 2 * NT - 1;
  constexpr int kLanesPerRow = 2 * NT, kRowsPerPass = 64 / kLanesPerRow, kPasses = 16 / kRowsPerPass;
  LDS_AS const uint8_t* staged = (LDS_AS const uint8_t*)staged_p;
  LDS_AS uint8_t* out = (LDS_AS uint8_t*)rows_p;
  const int lane = threadIdx.x & 63, r = lane & 15, gq = lane >> 4;
  float cs[PER_COL ? NT : 1][4], cb[HAS_BIAS ? NT : 1][4];
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int col = 16 * j + 4 * gq;
    if constexpr (PER_COL) {
      const f32x4 v = *reinterpret_cast<LDS_AS const f32x4*>(staged + kStagedColScale + col * 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) cs[j][e] = v[e];
    }
    if constexpr (HAS_BIAS) {
      const u32x2 v = *reinterpret_cast<LDS_AS const u32x2*>(staged + kStagedBias + col * 2);
      cb[j][0] = __uint_as_float(v[0] << 16);
      cb[j][1] = __uint_as_float(v[0] & 0xffff0000u);
      cb[j][2] = __uint_as_float(v[1] << 16);
      cb[j][3] = __uint_as_float(v[1] & 0xffff0000u);
    }
  }
  const int rows = g.M - m_wave < 16 * MT ? g.M - m_wave : 16 * MT;
  uint16_t* cbase = reinterpret_cast<uint16_t*>(g.C) + batch * g.stride_c + (int64_t)m_wave * g.ldc;
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(cbase, 0, rows > 0 ? rows * (int)g.ldc * 2 : 0, 0x00020000);
  const int row_in_pass = lane / kLanesPerRow, chunk = lane % kLanesPerRow;
  const int n_out = n_wave + 8 * chunk, pitch = (int)g.ldc * 2;
  const int voff0 = n_out < g.N ? row_in_pass * pitch + n_out * 2 : 0x7fffffff;
  const int pass_step = n_out < g.N ? kRowsPerPass * pitch : 0;
  static_for<MT>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
    const float staged_ra = *reinterpret_cast<LDS_AS const float*>(staged + kStagedRowScale + (16 * i + r) * 4);
    const float ra = g.sa_mode == MI355Q_GS_PER_ROW ? staged_ra : scalars.sa;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      float v[4];
      // (one scale after the other: their product can leave fp32's range where neither sums nor results do)
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = __builtin_fmaf(acc[i][j][e] * ra, PER_COL ? cs[PER_COL ? j : 0][e] : scalars.sb, HAS_BIAS ? cb[HAS_BIAS ? j : 0][e] : 0.0f);
      const int slot = (4 * j + gq) ^ (2 * ((r >> kShift) & kMask));
      *reinterpret_cast<LDS_AS u32x2*>(out + i * 16 * kRow + r * kRow + slot * 8) = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
    }
  });
  // (a wave reads only what it wrote itself, and its LDS instructions execute in order)
  static_for<MT>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
#pragma unroll
    for (int p = 0; p < kPasses; ++p) {
      const int row = p * kRowsPerPass + row_in_pass;
      const u32x4 o = *reinterpret_cast<LDS_AS const u32x4*>(out + i * 16 * kRow + row * kRow + ((chunk ^ ((row >> kShift) & kMask)) << 4));
      __builtin_amdgcn_raw_buffer_store_b128(o, rsrc, voff0 + (i * kPasses + p) * pass_step, 0, 2);  // aux 2: nontemporal
    }
  });
}

// The kernel's epilogues, GemmArgs::fast_epi of its launch.
enum RingEpilogue { kRingAny = 0, kRingFast = 1, kRingRows = 2 };

// Whether ring_epilogue_rows serves a launch: rows of C and of the accumulate input in aligned pieces of four, at offsets
// below 2^30 from a tile's first row.
inline bool ring_rows_ok(const GemmArgs& g, int64_t batches) {
  const int64_t es = g.out_bf16 ? 2 : 4;
  const auto pieces = [&](const void* p, int64_t ld, int64_t stride) {
    return reinterpret_cast<uintptr_t>(p) % (size_t)(4 * es) == 0 && ld >= 0 && ld % 4 == 0 && ld <= (int64_t(1) << 21) && (batches == 1 || stride % 4 == 0);
  };
  return g.N % 4 == 0 && g.N <= (1 << 21) && g.bias_mode != MI355Q_BIAS_FULL && pieces(g.C, g.ldc, g.stride_c) && (g.D == nullptr || pieces(g.D, g.ldd, g.stride_d));
}

// fp32 output, an accumulate input (or a full bias in its place), scales per column of A or row of B: the wave's sums go to LDS as
// they are, with the scales of a row behind it, and come back with a lane owning four columns of a row, whose accumulate input it
// has requested eight rows ahead.  Bound by the rows of C and D.  Column by column, each with a test and an address of its own as
// in ring_epilogue_any, the input cost a tile of 256 rows 33 us (us a product, that form -> this one: 4096 x 4096 x 14336 with an
// accumulate input 436 -> 213, fp32 258 -> 213, both 464 -> 244; 192 x 4096 x 14336 42.1 -> 22.7, 27.5 -> 21.7, 42.3 -> 23.2;
// 16 x 4096 x 4096 8.7 -> 7.4, 7.6 -> 7.4, 8.8 -> 7.6).
template <int MT, int NT, bool F32, bool HAS_D>
__device__ __forceinline__ void ring_epilogue_rows(const GemmArgs& g, int64_t batch, f32x4 (&acc)[MT][NT], int m_wave, int n_wave,
                                                   float* rows_p, ScalarScales scalars) {
  constexpr int kPitch = 16 * NT + 4, kLanesPerRow = 4 * NT, kRowsPerPass = 64 / kLanesPerRow, kPasses = 16 * MT / kRowsPerPass;
  constexpr int kAhead = kPasses < 8 ? kPasses : 8, es = F32 ? 4 : 2;
  static_assert(kPasses % kAhead == 0, "whole groups of rows");
  typedef typename std::conditional<F32, u32x4, u32x2>::type Piece;
  LDS_AS float* rows = (LDS_AS float*)rows_p;
  const int lane = threadIdx.x & 63, r = lane & 15, gq = lane >> 4;
  const int left = g.M - m_wave < 16 * MT ? g.M - m_wave : 16 * MT;
  const int row0 = lane / kLanesPerRow, n = n_wave + (lane % kLanesPerRow) * 4;
  const bool inside = n < g.N;  // (the four columns are inside or outside together; outside: an offset no descriptor covers)
  const auto view = [&](const uint8_t* p, int64_t stride, int64_t ld) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p) + (batch * stride + (int64_t)m_wave * ld) * es, 0,
                                             left > 0 ? ((left - 1) * (int)ld + g.N) * es : 0, 0x00020000);
  };
  const __amdgpu_buffer_rsrc_t to = view(g.C, g.stride_c, g.ldc), from = view(HAS_D ? g.D : g.C, HAS_D ? g.stride_d : g.stride_c, HAS_D ? g.ldd : g.ldc);
  const int to0 = inside ? (row0 * (int)g.ldc + n) * es : 0x7fffffff, to_step = inside ? kRowsPerPass * (int)g.ldc * es : 0;
  const int from0 = inside ? (row0 * (int)g.ldd + n) * es : 0x7fffffff, from_step = inside ? kRowsPerPass * (int)g.ldd * es : 0;
  const auto fetch = [&](Piece (&d)[HAS_D ? kAhead : 1], int pass) {
    if constexpr (HAS_D) {
#pragma unroll
      for (int p = 0; p < kAhead; ++p) {
        if constexpr (F32) d[p] = __builtin_bit_cast(Piece, __builtin_amdgcn_raw_buffer_load_b128(from, from0 + (pass + p) * from_step, 0, 0));
        else d[p] = __builtin_bit_cast(Piece, __builtin_amdgcn_raw_buffer_load_b64(from, from0 + (pass + p) * from_step, 0, 0));
      }
    }
  };
  Piece d[HAS_D ? kAhead : 1];
  fetch(d, 0);
  const bool a_rows = g.sa_mode == MI355Q_GS_PER_ROW, b_rows = g.sb_mode == MI355Q_GS_PER_ROW;
  float sa_c[4], sb_c[4], bias_c[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int ne = inside ? n + e : g.N - 1;
    sa_c[e] = g.sa_mode == MI355Q_GS_PER_COL ? g.sa[ne] : scalars.sa;
    sb_c[e] = g.sb_mode == MI355Q_GS_PER_COL ? g.sb[ne] : scalars.sb;
    bias_c[e] = g.bias_mode == MI355Q_BIAS_ROW_VECTOR ? load_out_as_f32(g.bias + batch * g.stride_bias * es, ne, !F32) : 0.0f;
  }
#pragma unroll
  for (int t = 0; t < 16 * MT; t += 64) {
    const int row = t + lane, m = m_wave + row < g.M ? m_wave + row : g.M - 1;
    if (row < 16 * MT) {
      rows[row * kPitch + 16 * NT] = a_rows ? g.sa[m] : 1.0f;
      rows[row * kPitch + 16 * NT + 1] = b_rows ? g.sb[m] : 1.0f;
    }
  }
  static_for<MT>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
#pragma unroll
    for (int j = 0; j < NT; ++j) *reinterpret_cast<LDS_AS f32x4*>(rows + (16 * i + r) * kPitch + 16 * j + 4 * gq) = acc[i][j];
  });
#pragma unroll 1
  for (int pass = 0; pass < kPasses && pass * kRowsPerPass < left; pass += kAhead) {
    Piece next[HAS_D ? kAhead : 1];
    fetch(next, pass + kAhead);  // (rows past the last one touch no memory)
#pragma unroll
    for (int p = 0; p < kAhead; ++p) {
      LDS_AS const float* row = rows + ((pass + p) * kRowsPerPass + row0) * kPitch;
      const f32x4 a = *reinterpret_cast<LDS_AS const f32x4*>(row + (lane % kLanesPerRow) * 4);
      const f32x2 s = *reinterpret_cast<LDS_AS const f32x2*>(row + 16 * NT);
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float t = a[e] * (a_rows ? s[0] : sa_c[e]);
        v[e] = t * (b_rows ? s[1] : sb_c[e]) + bias_c[e];
        if constexpr (HAS_D) v[e] += F32 ? __uint_as_float(d[p][F32 ? e : 0]) : __uint_as_float(e & 1 ? d[p][e >> 1] & 0xffff0000u : d[p][e >> 1] << 16);
      }
      const int at = to0 + (pass + p) * to_step;
      if constexpr (F32) __builtin_amdgcn_raw_buffer_store_b128(u32x4{__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3])}, to, at, 0, 2);
      else __builtin_amdgcn_raw_buffer_store_b64(u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])}, to, at, 0, 2);  // aux 2: nontemporal
    }
    if constexpr (HAS_D) {
#pragma unroll
      for (int p = 0; p < kAhead; ++p) d[p] = next[p];
    }
  }
}

// Every other form (rows of C or D that are no aligned pieces of four, a full bias beside an accumulate input): the wave's sums go to
// LDS as they are, then a rolled loop takes four columns of a row per lane.
template <int MT, int NT>
__device__ __forceinline__ void ring_epilogue_any(const GemmArgs& g, int64_t batch, f32x4 (&acc)[MT][NT], int m_wave, int n_wave,
                                                  float* rows, ScalarScales scalars) {
  constexpr int kPitch = 16 * NT + 4, kLanesPerRow = 4 * NT, kRowsPerPass = 64 / kLanesPerRow;
  const int lane = threadIdx.x & 63, r = lane & 15, gq = lane >> 4;
  static_for<MT>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
#pragma unroll
    for (int j = 0; j < NT; ++j) *reinterpret_cast<f32x4*>(rows + (16 * i + r) * kPitch + 16 * j + 4 * gq) = acc[i][j];
  });
  const int es = g.out_bf16 ? 2 : 4;
  uint8_t* C = g.C + batch * g.stride_c * es;
  const uint8_t* D = g.D ? g.D + batch * g.stride_d * es : nullptr;
  const uint8_t* bias = g.bias ? g.bias + batch * g.stride_bias * es : nullptr;
  const int n = n_wave + (lane % kLanesPerRow) * 4;
  if (n >= g.N) return;
  float sa_c[4], sb_c[4], bias_c[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int ne = n + e < g.N ? n + e : g.N - 1;
    sa_c[e] = g.sa_mode == MI355Q_GS_PER_COL ? g.sa[ne] : scalars.sa;
    sb_c[e] = g.sb_mode == MI355Q_GS_PER_COL ? g.sb[ne] : scalars.sb;
    bias_c[e] = g.bias_mode == MI355Q_BIAS_ROW_VECTOR ? load_out_as_f32(bias, ne, g.out_bf16) : 0.0f;
  }
  const bool vec_ok = (n + 3 < g.N) && ((g.ldc * es) % (4 * es) == 0) && ((reinterpret_cast<uintptr_t>(C) + (size_t)n * es) % (4 * es) == 0);
  const bool a_rows = g.sa_mode == MI355Q_GS_PER_ROW, b_rows = g.sb_mode == MI355Q_GS_PER_ROW, full = g.bias_mode == MI355Q_BIAS_FULL;
  const int last = g.M - m_wave < 16 * MT ? g.M - m_wave : 16 * MT;
#pragma unroll 4
  for (int row = lane / kLanesPerRow; row < last; row += kRowsPerPass) {
    const int m = m_wave + row;
    const f32x4 a = *reinterpret_cast<const f32x4*>(rows + row * kPitch + (lane % kLanesPerRow) * 4);
    const float ra = a_rows ? g.sa[m] : 1.0f, rb = b_rows ? g.sb[m] : 1.0f;
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      // (one of ra and sa_c is exactly 1, likewise rb and sb_c)
      float t = a[e] * (a_rows ? ra : sa_c[e]);
      t = t * (b_rows ? rb : sb_c[e]);
      v[e] = t + bias_c[e];
    }
    if (full || D) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int ne = n + e < g.N ? n + e : g.N - 1;
        if (full) v[e] += load_out_as_f32(bias, (int64_t)m * g.ldbias + ne, g.out_bf16);
        if (D) v[e] += load_out_as_f32(D, (int64_t)m * g.ldd + ne, g.out_bf16);
      }
    }
    uint8_t* const to = C + ((int64_t)m * g.ldc + n) * es;
    if (g.out_bf16) {
      const uint32_t w0 = pack_bf16x2(v[0], v[1]), w1 = pack_bf16x2(v[2], v[3]);
      uint16_t* c16 = reinterpret_cast<uint16_t*>(to);
      if (vec_ok) {
        *reinterpret_cast<u32x2*>(to) = u32x2{w0, w1};
      } else {
        c16[0] = (uint16_t)w0;
        if (n + 1 < g.N) c16[1] = (uint16_t)(w0 >> 16);
        if (n + 2 < g.N) c16[2] = (uint16_t)w1;
        if (n + 3 < g.N) c16[3] = (uint16_t)(w1 >> 16);
      }
    } else if (vec_ok) {
      *reinterpret_cast<f32x4*>(to) = f32x4{v[0], v[1], v[2], v[3]};
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (n + e < g.N) reinterpret_cast<float*>(to)[e] = v[e];
    }
  }
}

// BM = 16: one row tile, in LDS with 16 more rows that nothing reads (each of the four loading waves brings a whole region).
template <int BM>
struct RingShape {
  static constexpr int kRows = BM < 32 ? 32 : BM;  // of A in LDS
  static constexpr int kWavesM = BM >= 128 ? 2 : 1, kWavesN = kRingWaves / kWavesM;
  static constexpr int MT = BM / kWavesM / 16, NT = kRingBN / kWavesN / 16;
  static constexpr int kStage = (kRows + kRingBN) * kBK, kOffB = kRows * kBK;
  static constexpr int kFit = (160 * 1024 - kRingWaves * kRingScaleBytes - 64) / kStage;
  static constexpr int kStages = kFit < 7 ? kFit : 7;
};

// The load side of a workgroup: four waves that do nothing else.
template <int BM, bool A_KMAJOR, bool B_KMAJOR>
struct RingProducer {
  using Shape = RingShape<BM>;
  static constexpr int R = Shape::kStages, kStage = Shape::kStage, kOffB = Shape::kOffB;
  using LoaderA = RingLoader<A_KMAJOR, Shape::kRows>;
  using LoaderB = RingLoader<B_KMAJOR, kRingBN>;
  static constexpr int kOps = LoaderA::kPerWave + LoaderB::kPerWave;
  static_assert((R - 1) * kOps <= 63, "vmcnt holds 6 bits");
  LoaderA la;
  LoaderB lb;
  uint32_t slot, ring;  // LDS addresses of the next stage's slot and of the ring
  int next, stages;     // the stage of K the loaders point at, and their number
  int last_k;           // k in the last stage of K

  __device__ __forceinline__ void select() {
    const int valid = next == stages - 1 ? last_k : kBK;
    la.select(valid);
    lb.select(valid);
  }
  // The next stage's loads; then the loaders move on (after the last stage of K comes the first).
  template <bool NT_B>
  __device__ __forceinline__ void issue_stage() {
    static_for<LoaderA::kPerWave>([&](auto ic) { la.template issue<decltype(ic)::value, false>(slot); });
    static_for<LoaderB::kPerWave>([&](auto ic) { lb.template issue<decltype(ic)::value, NT_B>(slot + kOffB); });
    slot = slot + kStage == ring + R * kStage ? ring : slot + kStage;
    la.base += (uint64_t)la.step;
    lb.base += (uint64_t)lb.step;
    const bool was_last = next == stages - 1;
    if (++next == stages) {
      next = 0;
      la.base -= (uint64_t)(la.step * stages);
      lb.base -= (uint64_t)(lb.step * stages);
    }
    if (last_k != kBK && (was_last || next == stages - 1)) select();
  }
  // Until at most `left` stages' loads of this wave are outstanding.
  __device__ __forceinline__ static void wait_upto(int left) {
    static_for<R>([&](auto nc) {
      constexpr int n = decltype(nc)::value, ops = n * kOps;
      if (left == n || (n == 0 && left < 0)) __builtin_amdgcn_s_waitcnt((ops & 15) | ((ops >> 4) << 14) | 0x0f70);
    });
  }
};

// RingLoader for an operand whose rows begin anywhere: its chunks go through registers, 16 bytes per lane from any address, and are
// stored in the places of LDS that the other loader's DMA would give them.  Only the last stage of K has chunks that are partly, or not at
// all, inside the operand: fetch_edge() takes those from its last 16 bytes, and trim_edge() shifts them and clears what lies past K.
// (Before it rows and columns past the edge read others, and the last chunk of a row of an operand that is not K-major reads up to 15 bytes into
// the next row: there is one, of 16 bytes at least and 16 bytes on at least.)
template <bool KMAJOR, int EXT>
struct RaggedLoader {
  using G = typename RingLoader<KMAJOR, EXT>::G;
  static constexpr int kCPR = G::kChunksPerRow, kRowsPerRegion = 64 / kCPR, kPerWave = RingLoader<KMAJOR, EXT>::kPerWave;
  typedef uint32_t Any __attribute__((ext_vector_type(4), aligned(1)));
  typedef const __attribute__((address_space(1))) uint8_t* Global;
  Global base;              // the next stage to fetch
  Global last16;            // the operand's last 16 bytes
  int64_t step;
  uint32_t at[kPerWave];    // a lane's offsets in a stage
  int limit[kPerWave];      // and their k in it
  u32x4 v[2][kPerWave];     // of two stages
  uint32_t out;             // where the lane's first chunk goes, from the start of the operand's tile in LDS

  // p, ld, valid, wave: as in RingLoader; last: the operand's last 16 bytes
  __device__ __forceinline__ void init(const uint8_t* p, int64_t ld, int valid, int wave, const uint8_t* last) {
    const uint64_t b = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b), hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(b >> 32));
    base = reinterpret_cast<Global>(((uint64_t)hi << 32) | lo);
    last16 = reinterpret_cast<Global>(reinterpret_cast<uint64_t>(last));
    step = KMAJOR ? kBK : (int64_t)kBK * ld;
    const int lane = threadIdx.x & 63;
    out = (uint32_t)(wave * kPerWave * 1024 + lane * 16);
#pragma unroll
    for (int i = 0; i < kPerWave; ++i) {
      const int row = (wave * kPerWave + i) * kRowsPerRegion + lane / kCPR;
      const int c16 = ((lane % kCPR) ^ G::swizzle(row)) * 16;
      // (rows and columns past the edge take others: their products are never stored)
      if constexpr (KMAJOR) at[i] = (uint32_t)((row < valid ? row : valid - 1) * (int)ld + c16);
      else at[i] = (uint32_t)(row * (int)ld + (c16 < valid ? c16 : 0));
      limit[i] = KMAJOR ? c16 : row;
    }
  }
  __device__ __forceinline__ static u32x4 load(Global p) { return *reinterpret_cast<const __attribute__((address_space(1))) Any*>(p); }
  template <int P, int I>
  __device__ __forceinline__ void fetch() { v[P][I] = load(base + at[I]); }
  // A chunk of the last stage, of valid_k k: how many of its bytes count, where it begins, and how far that is past the last 16 bytes.
  struct Edge {
    int inside, over;
    Global p;
  };
  template <int I>
  __device__ __forceinline__ Edge edge(Global from, int valid_k) const {
    Edge e;
    e.inside = KMAJOR ? valid_k - limit[I] : (limit[I] < valid_k ? 16 : 0);
    const Global p = e.inside > 0 ? from + at[I] : last16;
    e.p = p < last16 ? p : last16;
    e.over = (int)(p - e.p);
    return e;
  }
  template <int P, int I>
  __device__ __forceinline__ void fetch_edge(int valid_k) { v[P][I] = load(edge<I>(base, valid_k).p); }
  // and the same chunk once it has come (the loader points past its stage by then)
  template <int P, int I>
  __device__ __forceinline__ void trim_edge(int valid_k) {
    const Edge e = edge<I>(base - step, valid_k);
    u32x4 w = v[P][I];
    if (__builtin_amdgcn_ballot_w64(e.over > 0) != 0) {  // rare: the operand's last rows
      uint64_t w0 = ((uint64_t)w[1] << 32) | w[0], w1 = ((uint64_t)w[3] << 32) | w[2];
      const int s = 8 * e.over;
      w0 = s >= 64 ? w1 >> (s - 64) : (s > 0 ? (w0 >> s) | (w1 << (64 - s)) : w0);
      w1 = s >= 64 ? 0 : w1 >> s;
      w = u32x4{(uint32_t)w0, (uint32_t)(w0 >> 32), (uint32_t)w1, (uint32_t)(w1 >> 32)};
    }
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const int n = e.inside - 4 * d;
      const uint32_t part = (1u << ((8 * n) & 31)) - 1u;
      v[P][I][d] = w[d] & (n >= 4 ? 0xffffffffu : (n > 0 ? part : 0u));
    }
  }
  // straight into LDS (whole stages of rows that begin at whole dwords)
  template <int I>
  __device__ __forceinline__ void to_lds(uint32_t tile, int wave) const {
    const uint64_t b = reinterpret_cast<uint64_t>(base);
    const i32x4 rsrc = {(int)(uint32_t)b, (int)((uint32_t)(b >> 32) & 0xffffu), 0x7ffffff0, 0x00020000};
    const uint32_t dst = tile + (uint32_t)((wave * kPerWave + I) * 1024);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" : : "s"(dst), "v"(at[I]), "s"(rsrc) : "memory", "m0");
  }
  template <int P, int I>
  __device__ __forceinline__ void store(uint32_t tile) const { *reinterpret_cast<LDS_AS u32x4*>(tile + out + I * 1024) = v[P][I]; }
};

// The load side for such operands.  Two stages are on their way in registers; each chunk's register is stored to LDS and at once asked for
// the stage after next.  (One stage on its way: 1000 x 3000 x 5000 31 us, two: 27.2.)
template <int BM, bool A_KMAJOR, bool B_KMAJOR>
struct RaggedProducer {
  using Shape = RingShape<BM>;
  static constexpr int R = Shape::kStages, kStage = Shape::kStage, kOffB = Shape::kOffB;
  using LoaderA = RaggedLoader<A_KMAJOR, Shape::kRows>;
  using LoaderB = RaggedLoader<B_KMAJOR, kRingBN>;
  LoaderA la;
  LoaderB lb;
  uint32_t slot, ring;
  int next, stages, last_k;  // next: the stage the loaders point at

  template <int P, int STORE, int FETCH>  // 0 nothing, 1 a whole stage, 2 the last stage
  __device__ __forceinline__ void move() {
    const int last = last_k;
    static_for<LoaderA::kPerWave>([&](auto ic) { chunk<P, decltype(ic)::value, STORE, FETCH>(la, slot, last); });
    static_for<LoaderB::kPerWave>([&](auto ic) { chunk<P, decltype(ic)::value, STORE, FETCH>(lb, slot + kOffB, last); });
    if constexpr (STORE != 0) slot = slot + kStage == ring + R * kStage ? ring : slot + kStage;
    if constexpr (FETCH != 0) {
      la.base += la.step;
      lb.base += lb.step;
      ++next;
    }
  }
  template <int P, int I, int STORE, int FETCH, typename Loader>
  __device__ __forceinline__ static void chunk(Loader& l, uint32_t tile, int last) {
    if constexpr (STORE == 2) l.template trim_edge<P, I>(last);
    if constexpr (STORE != 0) l.template store<P, I>(tile);
    if constexpr (FETCH == 1) l.template fetch<P, I>();
    if constexpr (FETCH == 2) l.template fetch_edge<P, I>(last);
  }
  template <int P>
  __device__ __forceinline__ void fetch_only() {
    if (next < stages - 1) move<P, 0, 1>();
    else if (next == stages - 1) move<P, 0, 2>();
  }
  // Stage s, in register set P = s % 2, to LDS; the stage after next into its place.
  template <int P>
  __device__ __forceinline__ void advance(int s) {
    if (next < stages - 1) move<P, 1, 1>();
    else if (next == stages - 1) move<P, 1, 2>();
    else if (s < stages - 1) move<P, 1, 0>();
    else if (s == stages - 1) move<P, 2, 0>();
  }
  // (the loads on their way stay there: only what was stored to LDS is waited for)
  __device__ __forceinline__ static void barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : : : "memory"); }
  __device__ __forceinline__ void run() {
    next = 0;
    fetch_only<0>();
    fetch_only<1>();
    advance<0>(0);
    barrier();  // the first stage is in LDS
    // stage s + 1 to LDS, into the slot of a stage that the consumers have had in their registers since the last barrier
    int s = 0;
    for (; s + 1 < stages; s += 2) {
      advance<1>(s + 1);
      barrier();
      advance<0>(s + 2);
      barrier();
    }
    if (s < stages) barrier();
  }
};

// The load side where rows begin at whole dwords, which is all that a load into LDS needs: every stage but the last comes that way,
// as in RingProducer.  The last one's chunks are asked for first of all and wait in registers for their turn.  (us, through registers
// / straight into LDS: 1000 x 3000 x 5000 27.2 / 25.3, 256 x 8188 x 8188 42.2 / 38.1, 64 x 4100 x 9996 22.2 / 21.9.)
template <int BM, bool A_KMAJOR, bool B_KMAJOR>
struct DwordProducer {
  using Shape = RingShape<BM>;
  static constexpr int R = Shape::kStages, kStage = Shape::kStage, kOffB = Shape::kOffB;
  using LoaderA = RaggedLoader<A_KMAJOR, Shape::kRows>;
  using LoaderB = RaggedLoader<B_KMAJOR, kRingBN>;
  static constexpr int kOps = LoaderA::kPerWave + LoaderB::kPerWave;
  LoaderA la;
  LoaderB lb;
  uint32_t slot, ring;
  int wave, stages, last_k;

  __device__ __forceinline__ void issue_stage() {
    static_for<LoaderA::kPerWave>([&](auto ic) { la.template to_lds<decltype(ic)::value>(slot, wave); });
    static_for<LoaderB::kPerWave>([&](auto ic) { lb.template to_lds<decltype(ic)::value>(slot + kOffB, wave); });
    slot = slot + kStage == ring + R * kStage ? ring : slot + kStage;
    la.base += la.step;
    lb.base += lb.step;
  }
  __device__ __forceinline__ void run() {
    const int whole = stages - 1;
    la.base += la.step * whole;
    lb.base += lb.step * whole;
    static_for<LoaderA::kPerWave>([&](auto ic) { la.template fetch_edge<0, decltype(ic)::value>(last_k); });
    static_for<LoaderB::kPerWave>([&](auto ic) { lb.template fetch_edge<0, decltype(ic)::value>(last_k); });
    la.base -= la.step * whole;
    lb.base -= lb.step * whole;
    for (int s = 0; s < R && s < whole; ++s) issue_stage();
    // (a stage's landing is what its barrier waits for; the last stage's chunks are older than any of them)
    RingProducer<BM, A_KMAJOR, B_KMAJOR>::wait_upto((whole < R ? whole : R) - 1);
    if (whole == 0) store_last();
    RaggedProducer<BM, A_KMAJOR, B_KMAJOR>::barrier();
    for (int s = 0; s < stages; ++s) {
      const bool more = s + R < whole;
      if (s + 1 == whole) store_last();
      else RingProducer<BM, A_KMAJOR, B_KMAJOR>::wait_upto(more ? R - 2 : whole - 2 - s);
      RaggedProducer<BM, A_KMAJOR, B_KMAJOR>::barrier();
      if (more) issue_stage();
    }
  }
  // the last stage into its slot (of a stage that the consumers are long done with); the loaders point past the stages before it
  __device__ __forceinline__ void store_last() {
    la.base += la.step;
    lb.base += lb.step;
    static_for<LoaderA::kPerWave>([&](auto ic) {
      la.template trim_edge<0, decltype(ic)::value>(last_k);
      la.template store<0, decltype(ic)::value>(slot);
    });
    static_for<LoaderB::kPerWave>([&](auto ic) {
      lb.template trim_edge<0, decltype(ic)::value>(last_k);
      lb.template store<0, decltype(ic)::value>(slot + kOffB);
    });
  }
};

// The multiply side.  Fragments are single-buffered as in gemm_tile16.h: those of the next stage replace this stage's as
// they die, so the barrier early in a stage finds every wave done with the stage's ring slot, and the next stage landed.
template <int BM, bool A_KMAJOR, bool B_KMAJOR, int FMT_A, int FMT_B>
struct RingConsumer {
  using Shape = RingShape<BM>;
  static constexpr int MT = Shape::MT, NT = Shape::NT, R = Shape::kStages, kStage = Shape::kStage;
  using ReaderA = RingReader<A_KMAJOR, Shape::kRows, MT>;
  using ReaderB = RingReader<B_KMAJOR, kRingBN, NT>;
  static constexpr int kBarrierAt = MT == 1 ? 0 : NT - 1;  // the stage's barrier stands in front of this MFMA, the first after which a fragment is dead
  f32x4 acc[MT][NT];
  i32x8 fa[MT], fb[NT];
  ReaderA ra;
  ReaderB rb;
  int rd;  // the ring slot the readers point at, in bytes

  template <int I>
  __device__ __forceinline__ void read_a() {
    static_for<ReaderA::kParts>([&](auto pc) { ra.template read<I, decltype(pc)::value, 0>(fa[I]); });
  }
  template <int J>
  __device__ __forceinline__ void read_b() {
    static_for<ReaderB::kParts>([&](auto pc) { rb.template read<J, decltype(pc)::value, 0>(fb[J]); });
  }
  __device__ __forceinline__ void first_fragments() {
    static_for<MT>([&](auto ic) { read_a<decltype(ic)::value>(); });
    static_for<NT>([&](auto jc) { read_b<decltype(jc)::value>(); });
  }
  // (after the last stage the reads fetch a slot whose contents are not used)
  __device__ __forceinline__ void stage() {
    static_for<MT * NT>([&](auto gc) {
      constexpr int gi = decltype(gc)::value, i = gi / NT, j = gi % NT;
      if constexpr (gi == kBarrierAt) {
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wave's reads of the stage are done
        __syncthreads();
        const int d = rd + kStage == R * kStage ? -(R - 1) * kStage : kStage;
        rd += d;
        ra.move(d);
        rb.move(d);
      }
      acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fb[j], fa[i], acc[i][j], mfma_code<FMT_B>(), mfma_code<FMT_A>(), 0, 0, 0, 0);
      if constexpr (j == NT - 1) read_a<i>();
      if constexpr (i == MT - 1) read_b<j>();
      __builtin_amdgcn_sched_barrier(0);
    });
  }
};

// NT_B: B is loaded with the nontemporal hint (ring_streams_b).  RAGGED: rows of A and B at any address, K of any length.
template <int BM, bool A_KMAJOR, bool B_KMAJOR, int FMT_A, int FMT_B, bool NT_B, bool RAGGED = false>
__global__ __launch_bounds__(kRingThreads) void fp8_gemm_ring_kernel(GemmArgs g, SplitArgs split) {
  using Producer = RingProducer<BM, A_KMAJOR, B_KMAJOR>;
  using Consumer = RingConsumer<BM, A_KMAJOR, B_KMAJOR, FMT_A, FMT_B>;
  using Shape = RingShape<BM>;
  constexpr int MT = Shape::MT, NT = Shape::NT, R = Shape::kStages;
  __shared__ __attribute__((aligned(1024))) uint8_t lds_ring[R * Shape::kStage];
  __shared__ __attribute__((aligned(16))) uint8_t lds_scales[kRingWaves * kRingScaleBytes];
  static_assert(kRingWaves * 16 * MT * (16 * NT + 4) * 4 <= R * Shape::kStage, "the epilogue's rows overlay the ring");

  // this workgroup's tile and part of K (whole stages)
  int tile_m = 0, tile_n, part = 0, tile;
  const int tiles = g.tiles_m * g.tiles_n;
  if (g.tiles_m == 1) {
    tile = blockIdx.x;
    if (split.parts > 1) {
      part = blockIdx.x / (unsigned)tiles;
      tile = blockIdx.x - part * tiles;
    }
    tile_n = tile;
  } else {
    // each XCD takes a contiguous range of (part, tile), so that the panels its workgroups share come out of its L2
    const int bid = blockIdx.x, units = gridDim.x;
    const int xcd = bid & 7, per = units >> 3, rem = units & 7;
    const int unit = (xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per) + (bid >> 3);
    part = split.parts > 1 ? unit / (unsigned)tiles : 0;
    tile = unit - part * tiles;
    tile_coords(tile, g.tiles_m, g.tiles_n, &tile_m, &tile_n);
  }
  if (split.parts > 1) {
    const unsigned all = (g.K + kBK - 1) / kBK;
    const int s0 = (int)(part * all / (unsigned)split.parts), s1 = (int)((part + 1) * all / (unsigned)split.parts);
    g.K = (g.K < s1 * kBK ? g.K : s1 * kBK) - s0 * kBK;
    g.A += (int64_t)s0 * kBK * (A_KMAJOR ? 1 : g.lda);
    g.B += (int64_t)s0 * kBK * (B_KMAJOR ? 1 : g.ldb);
  }
  const int m0 = tile_m * BM, n0 = tile_n * kRingBN;
  const int64_t batch = blockIdx.y;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int stages = (g.K + kBK - 1) / kBK;

  if (wave >= kRingWaves) {
    if constexpr (RAGGED) {
      const auto run = [&](auto& p) {
        p.slot = p.ring = (uint32_t)(uintptr_t)(LDS_AS uint8_t*)lds_ring;
        p.stages = stages;
        p.last_k = g.K - (stages - 1) * kBK;
        const uint8_t *a = g.A + batch * g.stride_a, *b = g.B + batch * g.stride_b;
        p.la.init(a + (int64_t)m0 * (A_KMAJOR ? g.lda : 1), g.lda, g.M - m0, wave - kRingWaves, a + (A_KMAJOR ? (g.M - 1) * g.lda + g.K : (g.K - 1) * g.lda + g.M) - 16);
        p.lb.init(b + (int64_t)n0 * (B_KMAJOR ? g.ldb : 1), g.ldb, g.N - n0, wave - kRingWaves, b + (B_KMAJOR ? (g.N - 1) * g.ldb + g.K : (g.K - 1) * g.ldb + g.N) - 16);
        p.run();
      };
      const uint64_t places = reinterpret_cast<uint64_t>(g.A) | reinterpret_cast<uint64_t>(g.B) | (uint64_t)(g.lda | g.ldb | g.stride_a | g.stride_b);
      if ((places & 3u) == 0) {
        DwordProducer<BM, A_KMAJOR, B_KMAJOR> p;
        p.wave = wave - kRingWaves;
        run(p);
      } else {
        RaggedProducer<BM, A_KMAJOR, B_KMAJOR> p;
        run(p);
      }
      return;
    }
    Producer p;
    p.slot = p.ring = (uint32_t)(uintptr_t)(LDS_AS uint8_t*)lds_ring;
    p.stages = stages;
    p.last_k = g.K - (stages - 1) * kBK;
    p.next = 0;
    p.la.init(g.A + batch * g.stride_a + (int64_t)m0 * (A_KMAJOR ? g.lda : 1), g.lda, g.M - m0, wave - kRingWaves);
    p.lb.init(g.B + batch * g.stride_b + (int64_t)n0 * (B_KMAJOR ? g.ldb : 1), g.ldb, g.N - n0, wave - kRingWaves);
    // With a K-major B in one row of tiles each strip walks K from a stage of its own and wraps around: strips in step send
    // requests that differ only in high address bits to the same few memory channels.  (An MN-major operand's ragged stage
    // has loads that go nowhere, which may retire ahead of older ones: it has to be the last, and nothing is counted then.)
    const bool tail_goes_nowhere = (!A_KMAJOR || !B_KMAJOR) && p.last_k != kBK;
    if (B_KMAJOR && g.tiles_m == 1 && !tail_goes_nowhere) {
      p.next = (int)((unsigned)tile_n * (unsigned)stages / (unsigned)g.tiles_n);
      p.la.base += (uint64_t)(p.la.step * p.next);
      p.lb.base += (uint64_t)(p.lb.step * p.next);
    }
    p.select();
    for (int s = 0; s < R && s < stages; ++s) p.template issue_stage<NT_B>();
    Producer::wait_upto(tail_goes_nowhere && stages <= R ? 0 : (stages < R ? stages : R) - 1);
    __syncthreads();  // the first stage is in LDS
    for (int s = 0; s < stages; ++s) {
      const bool more = s + R < stages;
      Producer::wait_upto(more ? R - 2 : (tail_goes_nowhere ? 0 : stages - 2 - s));
      __syncthreads();  // stage s + 1 is in LDS, and stage s in the consumers' registers
      if (more) p.template issue_stage<NT_B>();
    }
    return;
  }

  Consumer c;
  const int wm = (wave / Shape::kWavesN) * (16 * MT), wn = (wave % Shape::kWavesN) * (16 * NT);
  if (g.fast_epi == kRingFast) ScaleStager::issue<(MT + 1) / 2, NT / 2>(g, batch, m0 + wm, n0 + wn, reinterpret_cast<float*>(lds_scales + wave * kRingScaleBytes));
  const ScalarScales scalars = load_scalar_scales(g);
  const uint32_t ring = (uint32_t)(uintptr_t)(LDS_AS uint8_t*)lds_ring;
  c.ra.init(ring, wm);
  c.rb.init(ring + Producer::kOffB, wn);
  c.rd = 0;
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) c.acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  __syncthreads();
  c.first_fragments();
  for (int s = 0; s < stages; ++s) c.stage();

  // the producers have ended, and every load has landed; the ring is idle once the other consumers have read their last
  const int slot = (int)batch * tiles + tile, slots = tiles * gridDim.y;
  constexpr bool kPairs = BM >= 128;
  const uint32_t seen = !kPairs && split.parts > 1 ? split_look(split, slot) : 0;
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (split.parts > 1) {
    uint32_t* word = reinterpret_cast<uint32_t*>(lds_ring);
    if constexpr (kPairs) {
      if (!meet_in_pairs<4 * MT * NT, kRingWaves * 64>(
              split, slot, slots, part, word,
              [&](auto jc) { constexpr int j = decltype(jc)::value; return c.acc[j / (4 * NT)][j / 4 % NT][j % 4]; },
              [&](auto jc, float v) { constexpr int j = decltype(jc)::value; c.acc[j / (4 * NT)][j / 4 % NT][j % 4] = v; }))
        return;
    } else {
      if (threadIdx.x == 0) *word = seen;
      __syncthreads();
      const bool others_in = *word == (uint32_t)split.parts - 1;
      __syncthreads();
      // (rows past M travel too: whole lines of sums are stored and read faster than those of the rows that exist, 1 x 8192 x 1024
      // 8.1 us against 8.7 without them, 1 x 14336 x 4096 14.2 against 14.5)
      if (!split_exchange<4 * MT * NT, kRingWaves * 64>(
              split, slot, slots, part, true, others_in, word, [&](int j) { return c.acc[j / (4 * NT)][j / 4 % NT][j % 4]; },
              [&](int j, float v) { c.acc[j / (4 * NT)][j / 4 % NT][j % 4] = v; }))
        return;
    }
    __syncthreads();  // the word has been read
  }
  if (g.fast_epi == kRingFast) {
    const uint8_t* staged = lds_scales + wave * kRingScaleBytes;
    uint8_t* rows = lds_ring + wave * (16 * MT * 32 * NT);
    const bool per_col = g.sb_mode == MI355Q_GS_PER_COL, bias = g.bias_mode == MI355Q_BIAS_ROW_VECTOR;
    if (per_col && bias) ring_epilogue_fast<MT, NT, true, true>(g, batch, c.acc, m0 + wm, n0 + wn, staged, rows, scalars);
    else if (per_col) ring_epilogue_fast<MT, NT, true, false>(g, batch, c.acc, m0 + wm, n0 + wn, staged, rows, scalars);
    else if (bias) ring_epilogue_fast<MT, NT, false, true>(g, batch, c.acc, m0 + wm, n0 + wn, staged, rows, scalars);
    else ring_epilogue_fast<MT, NT, false, false>(g, batch, c.acc, m0 + wm, n0 + wn, staged, rows, scalars);
    return;
  }
  float* rows = reinterpret_cast<float*>(lds_ring) + wave * 16 * MT * (16 * NT + 4);
  if (g.fast_epi == kRingRows) {
    if (g.out_bf16 && g.D != nullptr) ring_epilogue_rows<MT, NT, false, true>(g, batch, c.acc, m0 + wm, n0 + wn, rows, scalars);
    else if (g.out_bf16) ring_epilogue_rows<MT, NT, false, false>(g, batch, c.acc, m0 + wm, n0 + wn, rows, scalars);
    else if (g.D != nullptr) ring_epilogue_rows<MT, NT, true, true>(g, batch, c.acc, m0 + wm, n0 + wn, rows, scalars);
    else ring_epilogue_rows<MT, NT, true, false>(g, batch, c.acc, m0 + wm, n0 + wn, rows, scalars);
  } else {
    ring_epilogue_any<MT, NT>(g, batch, c.acc, m0 + wm, n0 + wn, rows, scalars);
  }
}

// Whether B is loaded past the caches: every byte of it is read by one workgroup alone (one row of tiles, one product), and it is
// too large to be found in the memory-side cache by a later call.  Time without the hint over that with it, 1 to 128 rows, B [K, N]:
//   MiB          24    32    44    56    64    80    batches in all: 32    64    128   256   512
//   B cold       1.03  1.05  1.02  1.01  1.07  1.04                  1.09  1.08  1.07  1.05  1.06
//   B in there   0.85  0.93  0.87  0.95  0.93  0.86                  0.90  0.98  0.92  0.93  1.05
// So what decides is whether it is still there: of a matrix of more than a quarter of the cache a decoder's other layers leave
// nothing until its next turn, while a batch was mostly written just before.
inline bool ring_streams_b(const GemmArgs& g, int64_t batch) {
  if (g.tiles_m != 1 || (batch > 1 && g.stride_b == 0)) return false;
  const int64_t bytes = (int64_t)g.N * g.K;
  return bytes > (64LL << 20) || bytes > (256LL << 20) / batch;
}

template <int BM, bool AK, bool BK_, int FA, int FB>
void launch_ring(const GemmArgs& g, const SplitArgs& split, int64_t batch, hipStream_t st) {
  GemmArgs a = g;
  a.tiles_m = (g.M + BM - 1) / BM;
  a.tiles_n = (g.N + kRingBN - 1) / kRingBN;
  a.fast_epi = g.fast_epi && g.D == nullptr ? kRingFast : (ring_rows_ok(g, batch) ? kRingRows : kRingAny);
  dim3 grid((unsigned)(a.tiles_m * a.tiles_n * (split.parts > 1 ? split.parts : 1)), (unsigned)batch);
  if (ring_streams_b(a, batch)) fp8_gemm_ring_kernel<BM, AK, BK_, FA, FB, true><<<grid, kRingThreads, 0, st>>>(a, split);
  else fp8_gemm_ring_kernel<BM, AK, BK_, FA, FB, false><<<grid, kRingThreads, 0, st>>>(a, split);
}

// Operands at any alignment: A [M, K], either layout of B.  Without it they were copied into padded buffers first, a launch of its own
// that reads and writes both (ragged_plan in gemm_api.hip has figures and the rule).
template <int BM, bool BK_, int FA, int FB>
void launch_ring_ragged(const GemmArgs& g, const SplitArgs& split, int64_t batch, hipStream_t st) {
  GemmArgs a = g;
  a.tiles_m = (g.M + BM - 1) / BM;
  a.tiles_n = (g.N + kRingBN - 1) / kRingBN;
  a.fast_epi = g.fast_epi && g.D == nullptr ? kRingFast : (ring_rows_ok(g, batch) ? kRingRows : kRingAny);
  dim3 grid((unsigned)(a.tiles_m * a.tiles_n * (split.parts > 1 ? split.parts : 1)), (unsigned)batch);
  fp8_gemm_ring_kernel<BM, true, BK_, FA, FB, false, true><<<grid, kRingThreads, 0, st>>>(a, split);
}

}  // namespace mi355q
