// Which kernel serves which problem (split_plan in gemm_api.hip decides).
//
// 256 x 256 tiles move the fewest bytes from L2 into LDS per flop (four waves of 128 x 128 when the fast bf16 epilogue
// applies, see gemm_tile16.h, otherwise eight waves of 128 x 64).  Everything that does not fill the chip with them runs on
// the ring kernel, whose tiles have 16 to 256 rows and 128 columns, with K in parts where even its tiles leave compute
// units idle; and up to 16 rows against a large B [K, N] on the kernel that streams B into registers.
#pragma once
#include "gemm_ring.h"
#include "gemm_tile.h"
#include "gemm_tile16.h"

namespace mi355q {

// Tile columns to split off a 256 x 256 tiling whose last pass over the tiles would leave at least three quarters of the compute
// units idle (544 tiles on 256 CUs: two full passes and one of 32 tiles).  Those last columns then run as a second launch with the
// ring's 256 x 128 tiles, twice as many for about 0.6 of the time each (without -> with: 4096 x 4096 x 8704 126 -> 116 us, with an
// accumulate input 150 -> 139; 4096 x 2048 x 8448 73.7 -> 70.2; 8704 x 2048 x 8192, 1088 tiles, 125 -> 123).  A last pass that is more
// than a quarter full is left alone: the second launch then needs a pass of its own as long as what it saves.  0: no split.
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
  if (g.sa_mode == MI355Q_GS_PER_COL) t.sa = g.sa + n_off;
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
  else launch_tile<AK, BK_, FA, FB>(g, batch, st);
}

template <bool AK, bool BK_, int FA, int FB>
void launch_by_kind(const GemmArgs& g, const SplitArgs& split, int64_t batch, hipStream_t st) {
  if constexpr (AK) {
    if (split.kind == GemmKind::kRing16) return launch_ring<16, AK, BK_, FA, FB>(g, split, batch, st);
    if (split.kind == GemmKind::kRing32) return launch_ring<32, AK, BK_, FA, FB>(g, split, batch, st);
    if (split.kind == GemmKind::kRing64) return launch_ring<64, AK, BK_, FA, FB>(g, split, batch, st);
    if (split.kind == GemmKind::kRing192) return launch_ring<192, AK, BK_, FA, FB>(g, split, batch, st);
  }
  if (split.kind == GemmKind::kRing128) return launch_ring<128, AK, BK_, FA, FB>(g, split, batch, st);
  if (split.kind == GemmKind::kRing256) return launch_ring<256, AK, BK_, FA, FB>(g, split, batch, st);
  const int64_t c = tail_tile_columns(g.M, g.N, batch);
  if (c == 0) return launch_256x256<AK, BK_, FA, FB>(g, batch, st);
  const int64_t n_main = ((g.N + 255) / 256 - c) * 256;
  GemmArgs head = g;
  head.N = (int)n_main;
  head.fast_epi = epilogue_fast_ok(head, batch);
  launch_256x256<AK, BK_, FA, FB>(head, batch, st);
  launch_ring<256, AK, BK_, FA, FB>(columns_from<BK_>(g, n_main, batch), split, batch, st);
}

// One translation unit per operand layout instantiates this (gemm_inst_*.hip).
template <bool AK, bool BK_>
void launch_by_format(const GemmArgs& g, const SplitArgs& split, int fmt_a, int fmt_b, int64_t batch, hipStream_t st) {
  if (fmt_a == MI355Q_E4M3FN && fmt_b == MI355Q_E4M3FN) launch_by_kind<AK, BK_, MI355Q_E4M3FN, MI355Q_E4M3FN>(g, split, batch, st);
  else if (fmt_a == MI355Q_E4M3FN) launch_by_kind<AK, BK_, MI355Q_E4M3FN, MI355Q_E5M2>(g, split, batch, st);
  else if (fmt_b == MI355Q_E4M3FN) launch_by_kind<AK, BK_, MI355Q_E5M2, MI355Q_E4M3FN>(g, split, batch, st);
  else launch_by_kind<AK, BK_, MI355Q_E5M2, MI355Q_E5M2>(g, split, batch, st);
}

// Operands at any alignment (gemm_ragged_*.hip): A [M, K] on the ring kernel alone.
template <bool BK_, int FA, int FB>
void launch_ragged_by_kind(const GemmArgs& g, const SplitArgs& split, int64_t batch, hipStream_t st) {
  if (split.kind == GemmKind::kRing16) launch_ring_ragged<16, BK_, FA, FB>(g, split, batch, st);
  else if (split.kind == GemmKind::kRing32) launch_ring_ragged<32, BK_, FA, FB>(g, split, batch, st);
  else if (split.kind == GemmKind::kRing64) launch_ring_ragged<64, BK_, FA, FB>(g, split, batch, st);
  else if (split.kind == GemmKind::kRing128) launch_ring_ragged<128, BK_, FA, FB>(g, split, batch, st);
  else if (split.kind == GemmKind::kRing192) launch_ring_ragged<192, BK_, FA, FB>(g, split, batch, st);
  else launch_ring_ragged<256, BK_, FA, FB>(g, split, batch, st);
}
template <bool BK_>
void launch_ragged_by_format(const GemmArgs& g, const SplitArgs& split, int fmt_a, int fmt_b, int64_t batch, hipStream_t st) {
  if (fmt_a == MI355Q_E4M3FN && fmt_b == MI355Q_E4M3FN) launch_ragged_by_kind<BK_, MI355Q_E4M3FN, MI355Q_E4M3FN>(g, split, batch, st);
  else if (fmt_a == MI355Q_E4M3FN) launch_ragged_by_kind<BK_, MI355Q_E4M3FN, MI355Q_E5M2>(g, split, batch, st);
  else if (fmt_b == MI355Q_E4M3FN) launch_ragged_by_kind<BK_, MI355Q_E5M2, MI355Q_E4M3FN>(g, split, batch, st);
  else launch_ragged_by_kind<BK_, MI355Q_E5M2, MI355Q_E5M2>(g, split, batch, st);
}
void launch_gemm_ragged_kk(const GemmArgs& g, const SplitArgs& split, int fmt_a, int fmt_b, int64_t batch, hipStream_t st);
void launch_gemm_ragged_km(const GemmArgs& g, const SplitArgs& split, int fmt_a, int fmt_b, int64_t batch, hipStream_t st);

// A K-major / B K-major etc.; defined in gemm_inst_*.hip
void launch_gemm_kk(const GemmArgs& g, const SplitArgs& split, int fmt_a, int fmt_b, int64_t batch, hipStream_t st);
void launch_gemm_km(const GemmArgs& g, const SplitArgs& split, int fmt_a, int fmt_b, int64_t batch, hipStream_t st);
void launch_gemm_mk(const GemmArgs& g, const SplitArgs& split, int fmt_a, int fmt_b, int64_t batch, hipStream_t st);
void launch_gemm_mm(const GemmArgs& g, const SplitArgs& split, int fmt_a, int fmt_b, int64_t batch, hipStream_t st);

// K-major A, MN-major B, few rows; defined in gemm_stream.hip
void launch_gemm_stream(const GemmArgs& g, int fmt_a, int fmt_b, const SplitPlan& p, const SplitArgs& split, int64_t batch, hipStream_t st);

}  // namespace mi355q
