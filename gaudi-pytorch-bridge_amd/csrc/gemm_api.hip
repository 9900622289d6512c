// fp8_gemm_v2 C entry point: argument checks, kernel choice, and the any-shape
// fallback kernel.  The MFMA tile kernels live in gemm_tile.h.
#include <algorithm>
#include <cmath>

#include "gemm_dispatch.h"

namespace mi355q {

// Any shape, any stride, any alignment: one thread per element of C.  Slow;
// only for problems the tiled kernel's alignment rules exclude.
template <int FMT_A, int FMT_B>
__global__ __launch_bounds__(256) void fp8_gemm_simple_kernel(GemmArgs g, int64_t a_sm, int64_t a_sk,
                                                              int64_t b_sk, int64_t b_sn) {
  const int n = blockIdx.x * 16 + (threadIdx.x & 15);
  const int m = blockIdx.y * 16 + (threadIdx.x >> 4);
  const int64_t batch = blockIdx.z;
  if (m >= g.M || n >= g.N) return;
  const uint8_t* A = g.A + batch * g.stride_a + (int64_t)m * a_sm;
  const uint8_t* B = g.B + batch * g.stride_b + (int64_t)n * b_sn;
  float acc = 0.0f;
  for (int k = 0; k < g.K; ++k)
    acc += cvt_f32x1<FMT_A>(A[(int64_t)k * a_sk]) * cvt_f32x1<FMT_B>(B[(int64_t)k * b_sk]);
  float sa = 1.0f, sb = 1.0f;
  if (g.sa_mode == MI355Q_GS_HOST) sa = g.sa_host;
  else if (g.sa_mode == MI355Q_GS_DEV) sa = g.sa[0];
  else if (g.sa_mode == MI355Q_GS_PER_ROW) sa = g.sa[m];
  else if (g.sa_mode == MI355Q_GS_PER_COL) sa = g.sa[n];
  if (g.sb_mode == MI355Q_GS_HOST) sb = g.sb_host;
  else if (g.sb_mode == MI355Q_GS_DEV) sb = g.sb[0];
  else if (g.sb_mode == MI355Q_GS_PER_ROW) sb = g.sb[m];
  else if (g.sb_mode == MI355Q_GS_PER_COL) sb = g.sb[n];
  float t = acc * sa;
  t = t * sb;
  const int es = g.out_bf16 ? 2 : 4;
  if (g.bias_mode != MI355Q_BIAS_NONE) {
    const uint8_t* bias = g.bias + batch * g.stride_bias * es;
    const int64_t bo = g.bias_mode == MI355Q_BIAS_FULL ? (int64_t)m * g.ldbias + n : n;
    t += g.out_bf16 ? bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(bias)[bo])
                    : reinterpret_cast<const float*>(bias)[bo];
  }
  if (g.D) {
    const uint8_t* D = g.D + batch * g.stride_d * es;
    const int64_t d_o = (int64_t)m * g.ldd + n;
    t += g.out_bf16 ? bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(D)[d_o])
                    : reinterpret_cast<const float*>(D)[d_o];
  }
  uint8_t* C = g.C + batch * g.stride_c * es;
  const int64_t co = (int64_t)m * g.ldc + n;
  if (g.out_bf16) reinterpret_cast<uint16_t*>(C)[co] = (uint16_t)(pack_bf16x2(t, t) & 0xffffu);
  else reinterpret_cast<float*>(C)[co] = t;
}

// ------------------------------------------------------------------- dispatch

inline bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// The tiled kernels move 16-byte chunks: each operand's leading dimension,
// batch stride and base address must be multiples of 16 bytes, and so must K
// where K is an operand's contiguous dimension (a chunk is either all inside K
// or all outside).  Where m or n is contiguous, the chunk that straddles the
// extent brings in bytes of the row's padding (ld >= extent rounded up): those
// columns only feed outputs that are never stored.
inline bool k_chunks_ok(int trans_a, int trans_b, int64_t K) {
  return K % 16 == 0 || (trans_a && !trans_b);
}
inline bool tiled_ok(const void* A, int trans_a, int64_t lda, const void* B, int trans_b,
                     int64_t ldb, int64_t M, int64_t N, int64_t K, int64_t stride_a,
                     int64_t stride_b) {
  if (!al16(A) || !al16(B) || lda % 16 || ldb % 16 || stride_a % 16 || stride_b % 16) return false;
  if (!k_chunks_ok(trans_a, trans_b, K)) return false;
  // a stage of the tiled kernels spans up to 256 rows of ld bytes, addressed with 31-bit offsets
  if (lda > (1LL << 22) || ldb > (1LL << 22)) return false;
  return M > 0 && N > 0 && K > 0;
}

// What a launch takes on the ring kernel, in microseconds.
//  fixed          prologue, first loads, epilogue;
//  stage, busy    a stage of 128 k alone on the chip, and what comes on top where every compute unit has a workgroup;
//  round          the share of a stage that each further round of workgroups adds;
//  meet, level, crowd   the parts' meeting: fixed, per doubling of the parts, and on a full chip.
struct RingCost {
  GemmKind kind;
  int rows;
  double fixed, stage, busy, meet, level, crowd, round;
};
// Least-squares fits to 480 products (1 to 4096 rows, K from 512 to 16384, N from 256 to 28672, both layouts of B, whole and
// in 2 to 24 parts), each timed with the weights hot in the caches and cold and counted half and half.  The choice they make is
// 1.8 % slower in the mean than the best one measured, and 2.5 % over 240 other products of the
// same ranges.  The line of the 256-row tile is lowered by a tenth, which changed none of the 240
// choices.  The line of the 192-row tile lies between its neighbours' and a little above where they would meet: without it the 240
// take 3.0 %; of the 19 it is chosen for 16 are 1 to 20 % faster than on what would be chosen else, 3 slower (129 x 8992 x 7888 40 us
// against 31 on two parts of 128 rows).
constexpr RingCost kRingCosts[] = {
    {GemmKind::kRing16, 16, 2.84, 0.28, 0.44, 0.75, 0.83, 0.41, 1.10},
    {GemmKind::kRing32, 32, 3.18, 0.29, 0.26, 0.61, 1.29, 1.25, 1.34},
    {GemmKind::kRing64, 64, 3.99, 0.33, 0.16, -0.88, 2.86, 3.00, 1.35},
    {GemmKind::kRing128, 128, 4.99, 0.37, 0.22, -0.85, 3.75, 4.13, 1.22},
    {GemmKind::kRing192, 192, 5.79, 0.44, 0.20, -1.14, 4.39, 6.10, 1.28},
    {GemmKind::kRing256, 256, 6.59, 0.50, 0.19, -1.43, 5.03, 8.08, 1.19},
};

constexpr int kMostParts = 16;
// log2 of a number of parts.  (The choice is made twice on a call; with log2 and 64-bit divisions in the loop over the parts it
// took 1.1 us for 100 x 16384 x 256, without 0.33.)
constexpr double kLog2[kMostParts + 1] = {0.0, 0.0, 1.0, 1.5849625007211562, 2.0, 2.321928094887362, 2.584962500721156, 2.807354922057604, 3.0,
                                          3.169925001442312, 3.321928094887362, 3.4594316186372973, 3.584962500721156, 3.700439718141092,
                                          3.807354922057604, 3.9068905956085187, 4.0};

// The kernel and the cut that are expected to take least.
//  * Tiles of fewer than 128 rows exist for A [M, K]; up to 16 rows take the tile of 16, more of them none that is twice as high
//    as the product.
//  * At most one workgroup per compute unit where K is cut, parts of two stages at least, at most 16 of them.  Up to 128 rows
//    short products stay whole: below K = 1792 a cut of few strips gains a microsecond at most (1 x 1600 x 1024: 7.3 whole, 6.3
//    in four parts) and a cut of many loses as much; an A [K, M], whose tiles of 128 rows send all their sums, from 2304 on.
//  * 256 x 256 tiles take 1.42 us a stage in every pass over the compute units.
//  * From one of those per compute unit on, the table holds for the 192-row tile, and for the others only below one pass and a half
//    of them, with rows of A and B that start at whole 128-byte lines (a tile's rows of 128 bytes cross two lines otherwise, one of
//    256 x 256 three per two) and six stages or more.  us on the 256-row tile / on 256 x 256: 7341 x 896 x 2176 21.9 / 30.8, 3840 x 3712 x
//    6144 75.2 / 81.4, but 4096 x 4096 x 14336 204 / 173, 3636 x 2816 x 14752 171 / 147, 2409 x 3824 x 9600 119 / 112, 7836 x 512 x 3072 25.4 /
//    22.8.  With fp32 results it holds throughout, since 256 x 256 tiles run as eight waves there: 2048 x 1536 x 11008 48.5 / 58.0,
//    4096 x 8832 x 12672 376 / 396.
//  * Up to 16 rows against B [K, N] of more than 96 MiB: the stream kernel, whose 256-byte pieces of B come in at 5.5 TB/s
//    against 5.0 for the ring's 128 (16 x 8192 x 28672: 43.4 / 46.4 us; 16 x 8192 x 14336, 112 MiB, 26.4 / 26.3; 13 x 14144 x
//    5248, 71 MiB, 23.2 / 16.8).  Batches of 256 MiB and more in all, which the memory-side cache does not hold, take it too from
//    K = 2048 on (1 x 4096 x 4096, 25 of them 74 against 97; 100 of 1 x 2048 x 2048 82 against 90, but 1600 of 1 x 512 x 512 117 against
//    92; below, 12 of 1 x 4096 x 4096 37 against 34, but cold 38 against 50).  Its cut: a workgroup takes in its share of B at 37 GB/s,
//    or at its share of 6.5 TB/s where more of them run; no part shorter than 512, two turns of its eight waves.
SplitPlan split_plan(bool a_kmajor, int64_t lda, bool b_kmajor, int64_t ldb, int64_t M, int64_t N, int64_t K, int64_t batch, bool may_split,
                     bool fp32_rows, bool ring_only) {
  SplitPlan best;
  if (M <= 0 || N <= 0 || K <= 0 || batch <= 0) return best;
  const int64_t cus = compute_units(), stages = (K + kBK - 1) / kBK;
  best.batch = batch;
  // (the stream kernel addresses an operand with 31-bit offsets)
  const bool much = N * K > (96LL << 20) || (K >= 2048 && N * K >= (256LL << 20) / batch);
  if (!ring_only && a_kmajor && !b_kmajor && M <= 16 && much && K * ldb < 0x7fff0000LL && M * lda < 0x7fff0000LL) {
    best.kind = GemmKind::kStream;
    best.nb = 256;
    best.strips = (int)((N + 255) / 256);
    best.tile_rows = 16;
    const int64_t units = (K + 255) / 256, groups = best.strips * batch;
    double best_us = 0.0;
    for (int64_t parts = 1; parts <= 32 && (parts == 1 || (may_split && groups <= kMaxTickets && groups * parts <= 2 * cus && units / parts >= 2)); ++parts) {
      const double wgs = (double)(groups * parts), rate = std::min(37e3, 6.5e6 / std::min(wgs, (double)cus));
      double us = std::ceil(wgs / (double)cus) * (double)((units + parts - 1) / parts * 256) * 256.0 / rate;
      if (parts > 1) us += 0.5 + 0.2 * (double)parts + (double)M * (0.15 + 0.005 * (double)parts);
      if (parts > 1 && us >= best_us) continue;
      best_us = us;
      best.parts = (int)parts;
    }
    return best;
  }
  double best_us = 1e30;
  bool full_chip = false;
  if (!ring_only && M > 128 && N > 128) {
    const int64_t tiles = ((M + 255) / 256) * ((N + 255) / 256) * batch;
    best_us = (double)((tiles + cus - 1) / cus) * (double)stages * 1.42 + 6.0;
    full_chip = tiles >= cus && !fp32_rows && (2 * tiles >= 3 * cus || stages < 6 || lda % 128 != 0 || ldb % 128 != 0);
  }
  const double per_cu = 1.0 / (double)cus;
  for (const RingCost& c : kRingCosts) {
    if (a_kmajor ? (c.rows == 16) != (M <= 16) || (c.rows > 32 && c.rows >= 2 * M) : c.rows != 128 && c.rows != 256) continue;
    if (full_chip && c.rows != 192) continue;
    const int64_t tiles = ((M + c.rows - 1) / c.rows) * ((N + kRingBN - 1) / kRingBN), wgs = tiles * batch, rounds = (wgs + cus - 1) / cus;
    double fill = (double)std::min(wgs, cus) * per_cu;
    double in_stages = (double)stages * (c.stage + c.busy * fill) * (1.0 + (double)(rounds - 1) * c.round), us = c.fixed + in_stages;
    const bool in_parts = may_split && (M > 128 || K >= (a_kmajor ? 1792 : 2304));
    const int most = in_parts && stages >= 4 && rounds == 1 ? (int)std::min<int64_t>({cus / wgs, stages / 2, kMostParts}) : 1;
    for (int parts = 1; parts <= most; ++parts) {
      if (parts > 1) {
        fill = (double)(parts * (int)wgs) * per_cu;
        in_stages = (double)(((unsigned)stages + (unsigned)parts - 1) / (unsigned)parts) * (c.stage + c.busy * fill);
        us = c.fixed + in_stages + c.meet + c.level * kLog2[parts] + c.crowd * fill;
      }
      if (us >= best_us) continue;
      best_us = us;
      best.kind = c.kind;
      best.nb = kRingBN;
      best.strips = (int)tiles;
      best.parts = parts;
      best.tile_rows = c.rows;
      best.stages_us = in_stages;
    }
  }
  return best;
}

inline int64_t round_up16(int64_t v) { return (v + 15) & ~(int64_t)15; }
// The ring kernel's form and cut for operands that lie anywhere: those of aligned ones.
SplitPlan ragged_ring_plan(int trans_b, int64_t lda, int64_t ldb, int64_t M, int64_t N, int64_t K, int64_t batch, bool may_split) {
  return split_plan(true, round_up16(lda), trans_b != 0, round_up16(ldb), M, N, K, batch, may_split, false, true);
}

// Where the operands of a product of several matrices lie, for what depends on more than the pitches.
struct RaggedPlaces {
  const void *a, *b;
  int64_t stride_a, stride_b;
};

// The plan of a product whose operands lie anywhere (launch_gemm_ragged_*), A [M, K].  parts 0: not served, its operands are better copied
// first.  That is so where the copies end in 256 x 256 tiles, and where the loads' detour costs more than the copies would: it lengthens
// the stages by 0.3 for rows at whole dwords (DwordProducer), by 0.5 where only those of B are not and by 0.8 for others, and a copy is
// 4.6 us and twice the bytes at 5 TB/s.  Copied is what fp8_gemm_v2 would copy: an operand off the grid of 16 bytes, and both where K is
// off it, for they are filled up along K.  us a call with the copies / without: 1000 x 3000 x 5000 31.4 / 25.1, 16 x 8191 x 28671 122 / 65, 16 x
// 8191 x 28672 121 / 48, 64 x 4100 x 9999 38.1 / 23.9, 1 x 8191 x 20000 B [N, K] 87.7 / 51.6, 300 x 2049 x 1008 16.1 / 11.2, 1000 x 3008 x 5001 39.9 / 34.3,
// 256 x 8190 x 8192 51.8 / 41.5, but 1000 x 3001 x 5001 35.3 / 36.6, 3779 x 13824 x 1411 82.7 / 96.0; with A an odd byte from the grid 1000 x 3008 x 5008
// 29.5 / 34.0, 256 x 8192 x 8192 36.7 / 42.1, 300 x 2048 x 1024 11.5 / 10.2.  Of 150 such products the rule's way was never more than 5 % the slower.
// `at` nullptr: addresses and batch strides as aligned as the pitches, one matrix after the other; either: one of both will do.
SplitPlan ragged_plan(int trans_a, int64_t lda, int trans_b, int64_t ldb, int64_t M, int64_t N, int64_t K, int64_t batch, bool may_split,
                      const RaggedPlaces* at = nullptr, bool either = false) {
  SplitPlan none;
  none.parts = 0;
  if (trans_a || M < 1 || N < 16 || K < 256 || batch < 1 || lda > (1LL << 22) || ldb > (1LL << 22)) return none;
  // A chunk at the end of a row of B [K, N] is read into the next row, up to 15 bytes, so that one has to lie as far on.
  if (lda < 0 || ldb < (trans_b ? 0 : 16)) return none;
  if (split_plan(true, round_up16(lda), trans_b != 0, round_up16(ldb), M, N, K, batch, may_split).kind == GemmKind::kTile256) return none;
  const SplitPlan p = ragged_ring_plan(trans_b, lda, ldb, M, N, K, batch, may_split);
  const auto pays = [&](const RaggedPlaces& w) {
    const uint64_t a = reinterpret_cast<uint64_t>(w.a) | (uint64_t)(lda | (batch > 1 ? w.stride_a : 0));
    const uint64_t b = reinterpret_cast<uint64_t>(w.b) | (uint64_t)(ldb | (batch > 1 ? w.stride_b : 0));
    const double copied = (K % 16 != 0 || a % 16 != 0 ? (double)M * (double)K * (double)(w.stride_a == 0 ? 1 : batch) : 0.0) +
                          (K % 16 != 0 || b % 16 != 0 ? (double)N * (double)K * (double)(w.stride_b == 0 ? 1 : batch) : 0.0);
    return p.stages_us * (a % 4 != 0 ? 0.8 : (b % 4 != 0 ? 0.5 : 0.3)) < 4.6 + 0.4e-6 * copied;
  };
  const RaggedPlaces one_after_the_other{nullptr, nullptr, M * lda, (trans_b ? N : K) * ldb};
  return (at != nullptr && pays(*at)) || ((at == nullptr || either) && pays(one_after_the_other)) ? p : none;
}

// What launch_by_kind and launch_gemm_stream run; may_split: the caller brings the workspace.  A name gives the kernel and its
// tile (rows x columns x bytes of K per stage), with "split_" in front where K goes in parts.
const char* variant_name(int trans_a, int64_t lda, int trans_b, int64_t ldb, int64_t M, int64_t N, int64_t K, int64_t batch, bool may_split) {
  if (lda % 16 || ldb % 16 || lda > (1LL << 22) || ldb > (1LL << 22) || !k_chunks_ok(trans_a, trans_b, K)) return "simple";
  const SplitPlan p = split_plan(!trans_a, lda, trans_b != 0, ldb, M, N, K, batch, may_split);
  const bool cut = p.parts > 1;
  switch (p.kind) {
    case GemmKind::kStream: return cut ? "split_stream_16x256_registers_mfma16x16" : "stream_16x256_registers_mfma16x16";
    case GemmKind::kRing16: return cut ? "split_ring16x128x128_mfma16x16x128" : "ring16x128x128_mfma16x16x128";
    case GemmKind::kRing32: return cut ? "split_ring32x128x128_mfma16x16x128" : "ring32x128x128_mfma16x16x128";
    case GemmKind::kRing64: return cut ? "split_ring64x128x128_mfma16x16x128" : "ring64x128x128_mfma16x16x128";
    case GemmKind::kRing128: return cut ? "split_ring128x128x128_mfma16x16x128" : "ring128x128x128_mfma16x16x128";
    case GemmKind::kRing192: return cut ? "split_ring192x128x128_mfma16x16x128" : "ring192x128x128_mfma16x16x128";
    case GemmKind::kRing256: return cut ? "split_ring256x128x128_mfma16x16x128" : "ring256x128x128_mfma16x16x128";
    case GemmKind::kTile256: break;
  }
  return "tile256x256x128_mfma16x16x128";  // 32x32x64 with eight waves for epilogues beyond the fast bf16 one
}

}  // namespace mi355q

using namespace mi355q;

// mi355q_fp8_gemm_ws and mi355q_fp8_gemm_unaligned_ws (`unaligned`: ragged_plan decides, not tiled_ok).
static int gemm_call(const void* A, int fmt_a, int trans_a, int64_t lda, const void* B, int fmt_b,
                     int trans_b, int64_t ldb, void* C, int out_dtype, int64_t ldc, int64_t M,
                     int64_t N, int64_t K, const float* sa_dev, float sa_host, int sa_mode,
                     const float* sb_dev, float sb_host, int sb_mode, const void* bias,
                     int bias_mode, int64_t ldbias, const void* D, int64_t ldd, int64_t batch,
                     int64_t stride_a, int64_t stride_b, int64_t stride_c, int64_t stride_d,
                     int64_t stride_bias, void* workspace, size_t workspace_bytes, void* stream, bool unaligned) {
  auto fmt_ok = [](int f) { return f == MI355Q_E4M3FN || f == MI355Q_E5M2; };
  auto mode_ok = [](int m, const float* p) {
    if (m < MI355Q_GS_NONE || m > MI355Q_GS_PER_COL) return false;
    return !(m >= MI355Q_GS_DEV && p == nullptr);
  };
  if (!fmt_ok(fmt_a) || !fmt_ok(fmt_b)) return MI355Q_ERR_INVALID_ARGUMENT;
  if (out_dtype != MI355Q_F32 && out_dtype != MI355Q_BF16) return MI355Q_ERR_INVALID_ARGUMENT;
  if (M < 0 || N < 0 || K < 0 || batch < 0) return MI355Q_ERR_INVALID_ARGUMENT;
  if (!mode_ok(sa_mode, sa_dev) || !mode_ok(sb_mode, sb_dev)) return MI355Q_ERR_INVALID_ARGUMENT;
  if (bias_mode < MI355Q_BIAS_NONE || bias_mode > MI355Q_BIAS_FULL) return MI355Q_ERR_INVALID_ARGUMENT;
  if (bias_mode != MI355Q_BIAS_NONE && bias == nullptr) return MI355Q_ERR_INVALID_ARGUMENT;
  if (M == 0 || N == 0 || batch == 0) return MI355Q_OK;
  if (C == nullptr || (K > 0 && (A == nullptr || B == nullptr))) return MI355Q_ERR_INVALID_ARGUMENT;
  if (M > 0x7fffffffLL || N > 0x7fffffffLL || K > 0x7fffffffLL) return MI355Q_ERR_UNSUPPORTED;

  hipStream_t st = static_cast<hipStream_t>(stream);
  GemmArgs g;
  g.A = static_cast<const uint8_t*>(A);
  g.B = static_cast<const uint8_t*>(B);
  g.C = static_cast<uint8_t*>(C);
  g.lda = lda; g.ldb = ldb; g.ldc = ldc;
  g.M = (int)M; g.N = (int)N; g.K = (int)K;
  g.sa = sa_dev; g.sb = sb_dev; g.sa_host = sa_host; g.sb_host = sb_host;
  g.sa_mode = sa_mode; g.sb_mode = sb_mode;
  g.bias = static_cast<const uint8_t*>(bias);
  g.bias_mode = bias_mode; g.ldbias = ldbias;
  g.D = static_cast<const uint8_t*>(D);
  g.ldd = ldd;
  g.stride_a = stride_a; g.stride_b = stride_b; g.stride_c = stride_c; g.stride_d = stride_d;
  g.stride_bias = stride_bias;
  g.out_bf16 = out_dtype == MI355Q_BF16;
  g.fast_epi = 0;
  g.tiles_m = g.tiles_n = 0;

  const int64_t kMaxBatch = 65535;
  // Whether the call is served is settled here, on what either query was asked, and not by a piece of the batch or by the workspace.
  SplitPlan ragged;
  if (unaligned) {
    const RaggedPlaces at{A, B, stride_a, stride_b};
    ragged = ragged_plan(trans_a, lda, trans_b, ldb, M, N, K, batch, batch <= kMaxBatch, &at, true);
    if (ragged.parts == 0) return MI355Q_ERR_UNSUPPORTED;
    if (batch == 1) g.stride_a = g.stride_b = 0;  // (the kernel asks whether they are whole dwords)
  }
  for (int64_t b0 = 0; b0 < batch; b0 += kMaxBatch) {
    const int64_t nb = (batch - b0) < kMaxBatch ? (batch - b0) : kMaxBatch;
    GemmArgs gb = g;
    const int es = g.out_bf16 ? 2 : 4;
    gb.A = g.A + b0 * stride_a;
    gb.B = g.B + b0 * stride_b;
    gb.C = g.C + b0 * stride_c * es;
    if (g.D) gb.D = g.D + b0 * stride_d * es;
    if (g.bias) gb.bias = g.bias + b0 * stride_bias * es;
    // A full [M, N] bias and an accumulate input are the same kind of addend (out_dtype, added in
    // fp32 after the scales): alone, the bias takes D's place, which the fast epilogue knows.
    if (gb.bias_mode == MI355Q_BIAS_FULL && gb.D == nullptr) {
      gb.D = gb.bias;
      gb.ldd = gb.ldbias;
      gb.stride_d = gb.stride_bias;
      gb.bias = nullptr;
      gb.bias_mode = MI355Q_BIAS_NONE;
    }
    gb.fast_epi = epilogue_fast_ok(gb, nb);
    if (unaligned) {
      const bool as_asked = nb == batch && (workspace != nullptr || ragged.parts == 1);
      const SplitPlan plan = as_asked ? ragged : ragged_ring_plan(trans_b, lda, ldb, M, N, K, nb, false);
      SplitArgs split{plan.parts, nullptr, nullptr, plan.kind};
      if (plan.parts > 1) {
        if (!al16(workspace) || workspace_bytes < plan.workspace_bytes()) return MI355Q_ERR_WORKSPACE;
        split.tickets = static_cast<uint32_t*>(workspace);
        split.partials = reinterpret_cast<float*>(static_cast<uint8_t*>(workspace) + kTicketBytes);
      }
      if (trans_b) launch_gemm_ragged_kk(gb, split, fmt_a, fmt_b, nb, st);
      else launch_gemm_ragged_km(gb, split, fmt_a, fmt_b, nb, st);
    } else if (tiled_ok(gb.A, trans_a, lda, gb.B, trans_b, ldb, M, N, K, stride_a, stride_b)) {
      const bool ak = !trans_a, bk = trans_b != 0;
      // (K is walked in parts if the caller brought the room where they meet)
      // (fp32 results change the choice only where nothing is cut)
      const bool fp32_rows = !gb.out_bf16 && ring_rows_ok(gb, nb);
      const SplitPlan plan = split_plan(ak, lda, bk, ldb, M, N, K, nb, workspace != nullptr && nb == batch, fp32_rows);
      SplitArgs split{plan.parts, nullptr, nullptr};
      if (plan.parts > 1) {
        if (!al16(workspace) || workspace_bytes < plan.workspace_bytes()) return MI355Q_ERR_WORKSPACE;
        split.tickets = static_cast<uint32_t*>(workspace);
        split.partials = reinterpret_cast<float*>(static_cast<uint8_t*>(workspace) + kTicketBytes);
      }
      split.kind = plan.kind;
      if (plan.kind == GemmKind::kStream) launch_gemm_stream(gb, fmt_a, fmt_b, plan, split, nb, st);
      else if (ak && bk) launch_gemm_kk(gb, split, fmt_a, fmt_b, nb, st);
      else if (ak) launch_gemm_km(gb, split, fmt_a, fmt_b, nb, st);
      else if (bk) launch_gemm_mk(gb, split, fmt_a, fmt_b, nb, st);
      else launch_gemm_mm(gb, split, fmt_a, fmt_b, nb, st);
    } else {
      const int64_t a_sm = trans_a ? 1 : lda, a_sk = trans_a ? lda : 1;
      const int64_t b_sk = trans_b ? 1 : ldb, b_sn = trans_b ? ldb : 1;
      dim3 grid((unsigned)((N + 15) / 16), (unsigned)((M + 15) / 16), (unsigned)nb);
      if (grid.y > 65535u) return MI355Q_ERR_UNSUPPORTED;
      if (fmt_a == MI355Q_E4M3FN && fmt_b == MI355Q_E4M3FN) fp8_gemm_simple_kernel<MI355Q_E4M3FN, MI355Q_E4M3FN><<<grid, 256, 0, st>>>(gb, a_sm, a_sk, b_sk, b_sn);
      else if (fmt_a == MI355Q_E4M3FN) fp8_gemm_simple_kernel<MI355Q_E4M3FN, MI355Q_E5M2><<<grid, 256, 0, st>>>(gb, a_sm, a_sk, b_sk, b_sn);
      else if (fmt_b == MI355Q_E4M3FN) fp8_gemm_simple_kernel<MI355Q_E5M2, MI355Q_E4M3FN><<<grid, 256, 0, st>>>(gb, a_sm, a_sk, b_sk, b_sn);
      else fp8_gemm_simple_kernel<MI355Q_E5M2, MI355Q_E5M2><<<grid, 256, 0, st>>>(gb, a_sm, a_sk, b_sk, b_sn);
    }
    if (hipGetLastError() != hipSuccess) return MI355Q_ERR_LAUNCH;
  }
  return MI355Q_OK;
}

extern "C" {

const char* mi355q_fp8_gemm_variant(int trans_a, int64_t lda, int trans_b, int64_t ldb, int64_t M,
                                    int64_t N, int64_t K) {
  return variant_name(trans_a, lda, trans_b, ldb, M, N, K, 1, false);
}

const char* mi355q_fp8_gemm_ws_variant(int trans_a, int64_t lda, int trans_b, int64_t ldb, int64_t M,
                                       int64_t N, int64_t K, int64_t batch) {
  return variant_name(trans_a, lda, trans_b, ldb, M, N, K, batch, batch <= 65535);
}

size_t mi355q_fp8_gemm_workspace_bytes(int trans_a, int64_t lda, int trans_b, int64_t ldb, int64_t M, int64_t N, int64_t K,
                                       int64_t batch) {
  if (lda % 16 || ldb % 16 || !k_chunks_ok(trans_a, trans_b, K)) return 0;
  return batch > 65535 ? 0 : split_plan(!trans_a, lda, trans_b != 0, ldb, M, N, K, batch, true).workspace_bytes();
}

int mi355q_fp8_gemm(const void* A, int fmt_a, int trans_a, int64_t lda, const void* B, int fmt_b,
                    int trans_b, int64_t ldb, void* C, int out_dtype, int64_t ldc, int64_t M,
                    int64_t N, int64_t K, const float* sa_dev, float sa_host, int sa_mode,
                    const float* sb_dev, float sb_host, int sb_mode, const void* bias,
                    int bias_mode, int64_t ldbias, const void* D, int64_t ldd, int64_t batch,
                    int64_t stride_a, int64_t stride_b, int64_t stride_c, int64_t stride_d,
                    int64_t stride_bias, void* stream) {
  return mi355q_fp8_gemm_ws(A, fmt_a, trans_a, lda, B, fmt_b, trans_b, ldb, C, out_dtype, ldc, M, N, K, sa_dev, sa_host,
                            sa_mode, sb_dev, sb_host, sb_mode, bias, bias_mode, ldbias, D, ldd, batch, stride_a, stride_b,
                            stride_c, stride_d, stride_bias, nullptr, 0, stream);
}

int mi355q_fp8_gemm_unaligned_workspace_bytes(int trans_a, int64_t lda, int trans_b, int64_t ldb, int64_t M, int64_t N, int64_t K,
                                              int64_t batch, size_t* bytes) {
  if (bytes == nullptr) return MI355Q_ERR_INVALID_ARGUMENT;
  const SplitPlan p = ragged_plan(trans_a, lda, trans_b, ldb, M, N, K, batch, batch <= 65535);
  *bytes = p.parts == 0 ? 0 : p.workspace_bytes();
  return p.parts == 0 ? MI355Q_ERR_UNSUPPORTED : MI355Q_OK;
}

int mi355q_fp8_gemm_unaligned_query(const void* A, int trans_a, int64_t lda, int64_t stride_a, const void* B, int trans_b, int64_t ldb,
                                    int64_t stride_b, int64_t M, int64_t N, int64_t K, int64_t batch, size_t* bytes) {
  if (bytes == nullptr) return MI355Q_ERR_INVALID_ARGUMENT;
  const RaggedPlaces at{A, B, stride_a, stride_b};
  const SplitPlan p = ragged_plan(trans_a, lda, trans_b, ldb, M, N, K, batch, batch <= 65535, &at);
  *bytes = p.parts == 0 ? 0 : p.workspace_bytes();
  return p.parts == 0 ? MI355Q_ERR_UNSUPPORTED : MI355Q_OK;
}

int mi355q_fp8_gemm_ws(const void* A, int fmt_a, int trans_a, int64_t lda, const void* B, int fmt_b,
                       int trans_b, int64_t ldb, void* C, int out_dtype, int64_t ldc, int64_t M,
                       int64_t N, int64_t K, const float* sa_dev, float sa_host, int sa_mode,
                       const float* sb_dev, float sb_host, int sb_mode, const void* bias,
                       int bias_mode, int64_t ldbias, const void* D, int64_t ldd, int64_t batch,
                       int64_t stride_a, int64_t stride_b, int64_t stride_c, int64_t stride_d,
                       int64_t stride_bias, void* workspace, size_t workspace_bytes, void* stream) {
  return gemm_call(A, fmt_a, trans_a, lda, B, fmt_b, trans_b, ldb, C, out_dtype, ldc, M, N, K, sa_dev, sa_host, sa_mode, sb_dev, sb_host,
                   sb_mode, bias, bias_mode, ldbias, D, ldd, batch, stride_a, stride_b, stride_c, stride_d, stride_bias, workspace,
                   workspace_bytes, stream, false);
}

int mi355q_fp8_gemm_unaligned_ws(const void* A, int fmt_a, int trans_a, int64_t lda, const void* B, int fmt_b,
                                 int trans_b, int64_t ldb, void* C, int out_dtype, int64_t ldc, int64_t M,
                                 int64_t N, int64_t K, const float* sa_dev, float sa_host, int sa_mode,
                                 const float* sb_dev, float sb_host, int sb_mode, const void* bias,
                                 int bias_mode, int64_t ldbias, const void* D, int64_t ldd, int64_t batch,
                                 int64_t stride_a, int64_t stride_b, int64_t stride_c, int64_t stride_d,
                                 int64_t stride_bias, void* workspace, size_t workspace_bytes, void* stream) {
  return gemm_call(A, fmt_a, trans_a, lda, B, fmt_b, trans_b, ldb, C, out_dtype, ldc, M, N, K, sa_dev, sa_host, sa_mode, sb_dev, sb_host,
                   sb_mode, bias, bias_mode, ldbias, D, ldd, batch, stride_a, stride_b, stride_c, stride_d, stride_bias, workspace,
                   workspace_bytes, stream, true);
}

}  // extern "C"
