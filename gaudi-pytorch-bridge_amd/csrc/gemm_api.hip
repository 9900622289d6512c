// fp8_gemm_v2 C entry point: argument checks, kernel choice, and the any-shape
// fallback kernel.  The MFMA tile kernels live in gemm_tile.h.
#include <algorithm>

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

// More than 128 rows: the tiles of gemm_tile_split.h, one workgroup per compute unit at most, where they are expected to beat
// the uncut launch.  The estimates (us; `fill` is the share of the compute units that have a workgroup) are least-squares fits
// to 590 products of 130 to 4000 rows, K from 1536 to 14336 and N from 64 to 8192, whole and in 2 to 16 parts, each timed with
// the weights hot in the caches and cold and counted half and half, since a cut hides the cold weights' latency but costs the
// same meeting when they are hot: 500 x 3072 x 2048 takes 13.2 / 23.8 whole, 14.8 / 18.4 in two parts, 20.9 / 21.1 in four.
// Most are within 10 %.  The meeting costs more the fuller the chip is.  Beyond 16 parts nothing was faster.
SplitPlan tile_split_plan(int64_t M, int64_t N, int64_t K, int64_t batch) {
  SplitPlan best;
  const int64_t cus = compute_units(), pairs = (K + 2 * kBK - 1) / (2 * kBK);
  const TileChoice whole = N > 128 ? choose_tiles(M, N, K, batch) : TileChoice::k128x128;
  if (whole == TileChoice::k256x256 && ((M + 255) / 256) * ((N + 255) / 256) * batch >= cus) return best;
  auto tiles_of = [&](int64_t bm) { return ((M + bm - 1) / bm) * ((N + 127) / 128) * batch; };
  const double all_stages = (double)((K + kBK - 1) / kBK);
  double best_us = 0.85 * tile_us(whole, M, N, K, batch);
  if (whole == TileChoice::k128x128) best_us = all_stages * (0.52 + 0.29 * (double)tiles_of(128) / (double)cus) + 2.7;
  if (whole == TileChoice::k256x128) best_us = all_stages * 0.83 + 2.7 + (all_stages * 0.07 + 3.9) * (double)tiles_of(256) / (double)cus;
  for (const int64_t bm : {128, 256}) {
    const int64_t tiles = tiles_of(bm);
    for (int64_t parts = 2; parts <= 16 && parts <= pairs && parts * tiles <= cus; ++parts) {
      const double stages = 2.0 * (double)((pairs + parts - 1) / parts), levels = std::log2((double)parts);
      const double fill = (double)(parts * tiles) / (double)cus;
      const double us = bm == 128 ? stages * (0.51 + 0.13 * fill) + levels * (3.0 - 0.84 * fill) + 7.3 * fill + 2.9
                                  : stages * (0.72 + 0.07 * fill) + levels * (5.8 - 0.82 * fill) + 9.1 * fill + 4.3;
      if (us >= best_us) continue;
      best_us = us;
      best.tile = bm == 128 ? SplitTile::k128x128 : SplitTile::k256x128;
      best.nb = 128;
      best.strips = (int)(tiles / batch);
      best.parts = (int)parts;
      best.tile_rows = bm;
      best.batch = batch;
    }
  }
  return best;
}

// The cut that is expected to take least.  More than 128 rows: tile_split_plan.  For fewer the figures (microseconds, bytes
// per microsecond) are fits to 60 problems of 1 to 128 rows, K from 2048 to 14336 and N from 1024 to 38400, most of which
// they meet within two microseconds:
//  * a workgroup takes in its share of B at 37 GB/s, or at its share of 6.5 TB/s where more of them run;
//  * in the strip kernel A's tile travels along (a quarter of its bytes count with a K-major B, half with the shorter
//    pieces of an MN-major one);
//  * fixed costs, and with more than one part the meeting: each part's sums out, and all of them into the last one.
// Short products stay whole where the meeting costs them more than the parts save.  Whole and in parts, us a launch,
// weights hot in the caches / cold:
//  * the strip kernel below K = 1792: 1 x 1280 x 512, B [N, K], 8.9 / 8.9 and 9.5 / 9.4; 8 x 1536 x 512 8.2 / 9.3 and 8.8 / 9.0
//    (2048: 8 x 2048 x 512 9.5 / 10.7 and 9.1 / 9.5);
//  * the stream kernel below K = 2048, against the strip kernel whole: 1 x 1024 x 2048 6.8 / 8.5 and 10.3 / 10.1;
//  * no part of the stream kernel shorter than 512, two turns of its eight waves, since in a part of 256 a wave's first
//    loads have none behind them: 8 x 2048 x 4096 in eight of those 12.1 / 12.0, in four parts on the strip kernel 10.0 / 10.2.
SplitPlan split_plan(bool a_kmajor, int64_t lda, bool b_kmajor, int64_t ldb, int64_t M, int64_t N, int64_t K, int64_t batch, bool may_split) {
  SplitPlan best;
  if (M <= 0 || N <= 0 || K <= 0 || batch <= 0) return best;
  if (M > 128) return may_split ? tile_split_plan(M, N, K, batch) : best;
  const double cus = (double)compute_units();
  double best_us = 0.0;
  auto consider = [&](bool stream, int64_t nb, int64_t tile_rows, int64_t unit) {
    const int64_t shortest = stream ? 512 : unit;  // part
    const bool in_parts = may_split && K >= (stream ? 2048 : 1792);
    const int64_t strips = (N + nb - 1) / nb, groups = strips * batch, units = (K + unit - 1) / unit;
    const int64_t rows = M < 32 && tile_rows <= 32 ? M : tile_rows;  // rows of sums that travel (those of one row tile alone can be left out)
    const double width = (double)nb + (stream ? 0.0 : (double)tile_rows * (b_kmajor ? 0.25 : 0.5));
    for (int64_t parts = 1; parts <= 32 && parts <= units; ++parts) {
      if (parts > 1 && (!in_parts || groups > kMaxTickets || (double)(groups * parts) > 2.0 * cus)) break;
      if (parts > 1 && (units + parts - 1) / parts * unit < shortest) break;
      const double wgs = (double)(groups * parts), rounds = std::ceil(wgs / cus);
      const double rate = std::min(37e3, 6.5e6 / std::min(wgs, cus));
      double us = rounds * (double)((units + parts - 1) / parts * unit) * width / rate + 4.5;
      if (parts > 1)
        us += stream ? 0.5 + 0.2 * (double)parts + (double)rows * (0.15 + 0.005 * (double)parts)
                     : 2.0 + 0.25 * (double)parts + ((double)parts + 1.5) * (double)(rows * nb * 4) / 50e3;
      if (best.nb != 0 && us >= best_us) continue;
      best_us = us;
      best.stream = stream;
      best.nb = (int)nb;
      best.strips = (int)strips;
      best.parts = (int)parts;
      best.tile_rows = tile_rows;
      best.batch = batch;
    }
  };
  // (the stream kernel addresses an operand with 31-bit offsets)
  if (a_kmajor && !b_kmajor && M <= 16 && K * ldb < 0x7fff0000LL && M * lda < 0x7fff0000LL) consider(true, 256, 16, 256);
  consider(false, 128, !a_kmajor ? 128 : (M <= 32 ? 32 : (M <= 64 ? 64 : 128)), kBK);
  return best;
}

// What launch_by_size and launch_gemm_stream run; may_split: the caller brings the workspace.
const char* variant_name(int trans_a, int64_t lda, int trans_b, int64_t ldb, int64_t M, int64_t N, int64_t K, int64_t batch, bool may_split) {
  if (lda % 16 || ldb % 16 || lda > (1LL << 22) || ldb > (1LL << 22) || !k_chunks_ok(trans_a, trans_b, K)) return "simple";
  const SplitPlan p = split_plan(!trans_a, lda, trans_b != 0, ldb, M, N, K, batch, may_split);
  if (M <= 128) {
    if (p.stream) return p.parts > 1 ? "split_stream_Mx256_registers_mfma16x16" : "stream_Mx256_registers_mfma16x16";
    return p.parts > 1 ? "split_strip_Mx128x128_ring_mfma32x32x64" : "strip_Mx128x128_ring_mfma32x32x64";
  }
  if (p.tile == SplitTile::k128x128) return "split_tile128x128x128_mfma32x32x64";
  if (p.tile == SplitTile::k256x128) return "split_tile256x128x128_mfma32x32x64";
  switch (N > 128 ? choose_tiles(M, N, K, batch) : TileChoice::k128x128) {
    case TileChoice::k256x256: return "tile256x256x128_mfma16x16x128";  // 32x32x64 with eight waves for epilogues beyond the fast bf16 one
    case TileChoice::k256x128: return "tile256x128x128_mfma32x32x64";
    case TileChoice::k128x128: break;
  }
  return "tile128x128x128_mfma32x32x64";
}

}  // namespace mi355q

using namespace mi355q;

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

int mi355q_fp8_gemm_ws(const void* A, int fmt_a, int trans_a, int64_t lda, const void* B, int fmt_b,
                       int trans_b, int64_t ldb, void* C, int out_dtype, int64_t ldc, int64_t M,
                       int64_t N, int64_t K, const float* sa_dev, float sa_host, int sa_mode,
                       const float* sb_dev, float sb_host, int sb_mode, const void* bias,
                       int bias_mode, int64_t ldbias, const void* D, int64_t ldd, int64_t batch,
                       int64_t stride_a, int64_t stride_b, int64_t stride_c, int64_t stride_d,
                       int64_t stride_bias, void* workspace, size_t workspace_bytes, void* stream) {
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
    if (tiled_ok(gb.A, trans_a, lda, gb.B, trans_b, ldb, M, N, K, stride_a, stride_b)) {
      const bool ak = !trans_a, bk = trans_b != 0;
      // (K is walked in parts if the caller brought the room where they meet)
      const SplitPlan plan = split_plan(ak, lda, bk, ldb, M, N, K, nb, workspace != nullptr && nb == batch);
      SplitArgs split{plan.parts, nullptr, nullptr};
      if (plan.parts > 1) {
        if (!al16(workspace) || workspace_bytes < plan.workspace_bytes()) return MI355Q_ERR_WORKSPACE;
        split.tickets = static_cast<uint32_t*>(workspace);
        split.partials = reinterpret_cast<float*>(static_cast<uint8_t*>(workspace) + kTicketBytes);
        split.tile = plan.tile;
      }
      if (plan.stream) launch_gemm_stream(gb, fmt_a, fmt_b, plan, split, nb, st);
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

}  // extern "C"
