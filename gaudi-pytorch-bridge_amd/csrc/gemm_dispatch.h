// Which kernel serves which problem.
//
// Above 128 rows there are three tiles, and tile_us() says what a product takes on each.  256 x 256 moves the fewest
// bytes from L2 into LDS per flop (four waves of 128 x 128 when the fast bf16 epilogue applies, see gemm_tile.h,
// otherwise eight waves of 128 x 64); 256 x 128 (four waves of 128 x 64: 1.5 KB of LDS fragments read per MFMA; as
// eight waves of 128 x 32 it read 2.5 KB and was 3 to 8 % slower at 256 x 8192 x 28672) has twice the tiles at 1.5
// times that traffic; 128 x 128 (eight waves) four times, and two workgroups of it fit a compute unit (80 KB of LDS and
// at most 128 registers each) and cover each other's waits.  What decides is the number of passes over the compute
// units: 1536 x 8192 x 8192 is 192 tiles of 256 x 256, one pass of 90 us, or 384 of 256 x 128, two passes of 65 us each.
// (A 4-wave kernel with two workgroups per CU and 64-byte K stages, meant to
// hide the epilogue behind the other workgroup's MFMAs, was measured against
// the 256 x 128 tiles: bound by its global->LDS traffic on large problems and
// no faster on these.)
// Where even the smaller tiles leave compute units idle, K is cut as well (gemm_tile_split.h, split_plan).
// Few rows of A (M <= 128) take the strip kernel, which streams B once through a
// deep ring.
#pragma once
#include <cmath>

#include "gemm_skinny.h"
#include "gemm_tile.h"
#include "gemm_tile16.h"
#include "gemm_tile_split.h"

namespace mi355q {

enum class TileChoice { k256x256, k256x128, k128x128 };

// What a launch of M > 128 rows takes on one kind of tile, in microseconds, without a split of K.  The figures are fits to
// 60 products of 129 to 3000 rows, K from 1024 to 16384 and N from 1024 to 28672 (most within 15 %): a stage of 128 k takes a
// workgroup 0.8 us as a 128 x 128 tile (1.25 us for two of them on a compute unit), 1.12 us as a 256 x 128 tile and 1.42
// us as a 256 x 256 tile, since a compute unit takes in no more than about 40 KB a microsecond of such panels.
inline double tile_us(TileChoice t, int64_t M, int64_t N, int64_t K, int64_t batch) {
  const double cus = compute_units(), stages = (double)((K + kBK - 1) / kBK);
  const int64_t bm = t == TileChoice::k128x128 ? 128 : 256, bn = t == TileChoice::k256x256 ? 256 : 128;
  const double tiles = (double)((M + bm - 1) / bm) * (double)((N + bn - 1) / bn) * (double)batch;
  if (t == TileChoice::k256x256) return std::ceil(tiles / cus) * stages * 1.42 + 6.0;
  if (t == TileChoice::k256x128) return std::ceil(tiles / cus) * stages * 1.12 + 5.0;
  const double full = std::floor(tiles / (2 * cus)), rest = tiles - full * 2 * cus;
  return stages * (full * 1.25 + (rest > cus ? 1.25 : (rest > 0 ? 0.8 : 0.0))) + 5.0;
}

// For M > 128 and N > 128.  (From one 256 x 256 tile per compute unit on nothing else was faster.)
inline TileChoice choose_tiles(int64_t M, int64_t N, int64_t K, int64_t batch) {
  if (((M + 255) / 256) * ((N + 255) / 256) * batch >= compute_units()) return TileChoice::k256x256;
  TileChoice best = TileChoice::k128x128;
  for (TileChoice t : {TileChoice::k256x128, TileChoice::k256x256})
    if (tile_us(t, M, N, K, batch) < tile_us(best, M, N, K, batch)) best = t;
  return best;
}

// Tile columns to split off a 256 x 256 tiling whose last pass over the tiles would
// leave at least three quarters of the compute units idle (320 tiles on 256
// CUs: one full pass and one of 64 tiles).  Those last columns then run as a second
// launch with 256 x 128 tiles, twice as many for about 0.6 of the time each
// (2048 x 10240 x 8192: 0.156 -> 0.145 ms).  With a last pass that is half
// full the second launch costs what it saves (4096 x 14336 x 4096: 0.177 ms
// either way), so those are left alone.  0: no split.
inline int64_t tail_tile_columns(int64_t M, int64_t N, int64_t batch) {
  const int64_t cus = compute_units();
  const int64_t tm = (M + 255) / 256, tn = (N + 255) / 256;
  const int64_t tiles = tm * tn;
  if (batch != 1 || tiles < cus) return 0;
  const int64_t tail = tiles % cus;
  if (tail == 0 || 4 * tail > cus) return 0;
  const int64_t c = (tail + tm - 1) / tm;  // whole tile columns that hold the tail
  // the rest must still be whole passes, and the split-off part must fit one pass of half tiles
  if (c >= tn || 2 * c * tm > cus + cus / 4) return 0;
  return c;
}

// The same problem restricted to columns [n_off, N) of B and C.
template <bool B_KMAJOR>
GemmArgs columns_from(const GemmArgs& g, int64_t n_off, int64_t batch) {
  GemmArgs t = g;
  const int es = g.out_bf16 ? 2 : 4;
  t.N = g.N - (int)n_off;
  t.B = g.B + (B_KMAJOR ? n_off * g.ldb : n_off);
  t.C = g.C + n_off * es;
  if (g.sb_mode == MI355Q_GS_PER_COL) t.sb = g.sb + n_off;
  if (g.bias_mode != MI355Q_BIAS_NONE) t.bias = g.bias + n_off * es;
  if (g.D) t.D = g.D + n_off * es;
  t.fast_epi = epilogue_fast_ok(t, batch);
  return t;
}

template <bool AK, bool BK_, int FA, int FB>
void launch_256x256(const GemmArgs& g, int64_t batch, hipStream_t st) {
  // the fast bf16 epilogue without an accumulate input: four waves on the 16x16x128 MFMA (gemm_tile16.h)
  if (g.fast_epi && g.D == nullptr) launch_tile16<AK, BK_, FA, FB>(g, batch, st);
  else launch_tile<256, 256, 4, false, AK, BK_, FA, FB>(g, batch, st);
}

template <bool AK, bool BK_, int FA, int FB>
void launch_by_size(const GemmArgs& g, const SplitArgs& split, int64_t batch, hipStream_t st) {
  if (split.tile == SplitTile::k128x128) {
    launch_tile_split<128, 128, 4, AK, BK_, FA, FB>(g, split, batch, st);
  } else if (split.tile == SplitTile::k256x128) {
    launch_tile_split<256, 128, 2, AK, BK_, FA, FB>(g, split, batch, st);
  } else if (g.M > 128 && g.N > 128) {
    switch (choose_tiles(g.M, g.N, g.K, batch)) {
      case TileChoice::k256x256: {
        const int64_t c = tail_tile_columns(g.M, g.N, batch);
        if (c == 0) {
          launch_256x256<AK, BK_, FA, FB>(g, batch, st);
        } else {
          const int64_t n_main = ((g.N + 255) / 256 - c) * 256;
          GemmArgs head = g;
          head.N = (int)n_main;
          head.fast_epi = epilogue_fast_ok(head, batch);
          launch_256x256<AK, BK_, FA, FB>(head, batch, st);
          launch_tile<256, 128, 2, false, AK, BK_, FA, FB>(columns_from<BK_>(g, n_main, batch), batch, st);
        }
        break;
      }
      case TileChoice::k256x128: launch_tile<256, 128, 2, false, AK, BK_, FA, FB>(g, batch, st); break;
      case TileChoice::k128x128: launch_tile<128, 128, 4, false, AK, BK_, FA, FB, 2>(g, batch, st); break;
    }
  } else if (g.M <= 128) {
    launch_skinny_by_m<AK, BK_, FA, FB>(g, split, batch, st);
  } else {
    launch_tile<128, 128, 4, false, AK, BK_, FA, FB, 2>(g, batch, st);
  }
}

// One translation unit per operand layout instantiates this (gemm_inst_*.hip).
template <bool AK, bool BK_>
void launch_by_format(const GemmArgs& g, const SplitArgs& split, int fmt_a, int fmt_b, int64_t batch, hipStream_t st) {
  if (fmt_a == MI355Q_E4M3FN && fmt_b == MI355Q_E4M3FN) launch_by_size<AK, BK_, MI355Q_E4M3FN, MI355Q_E4M3FN>(g, split, batch, st);
  else if (fmt_a == MI355Q_E4M3FN) launch_by_size<AK, BK_, MI355Q_E4M3FN, MI355Q_E5M2>(g, split, batch, st);
  else if (fmt_b == MI355Q_E4M3FN) launch_by_size<AK, BK_, MI355Q_E5M2, MI355Q_E4M3FN>(g, split, batch, st);
  else launch_by_size<AK, BK_, MI355Q_E5M2, MI355Q_E5M2>(g, split, batch, st);
}

// A K-major / B K-major etc.; defined in gemm_inst_*.hip
void launch_gemm_kk(const GemmArgs& g, const SplitArgs& split, int fmt_a, int fmt_b, int64_t batch, hipStream_t st);
void launch_gemm_km(const GemmArgs& g, const SplitArgs& split, int fmt_a, int fmt_b, int64_t batch, hipStream_t st);
void launch_gemm_mk(const GemmArgs& g, const SplitArgs& split, int fmt_a, int fmt_b, int64_t batch, hipStream_t st);
void launch_gemm_mm(const GemmArgs& g, const SplitArgs& split, int fmt_a, int fmt_b, int64_t batch, hipStream_t st);

// K-major A, MN-major B, few rows; defined in gemm_stream.hip
void launch_gemm_stream(const GemmArgs& g, int fmt_a, int fmt_b, const SplitPlan& p, const SplitArgs& split, int64_t batch, hipStream_t st);

}  // namespace mi355q
