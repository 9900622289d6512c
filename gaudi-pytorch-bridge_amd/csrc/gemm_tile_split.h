// The 128 x 128 and 256 x 128 tiles of gemm_tile.h with K in parts over workgroups, for products of more than 128 rows
// whose tiles leave compute units idle (256 x 14336 x 4096 is 64 tiles of 128 x 128 for 256 units: 104 us unsplit, 40 us
// in four parts).  What bounds them: a compute unit takes in about 40 KB of panels a microsecond, and on top the
// meeting, 2 to 3 us a level for 128 x 128 sums and 5 to 6 for 256 x 128, with 7 to 9 on top on a full chip (the fits that
// choose are in gemm_api.hip).  With two
// workgroups per compute unit the same product takes 47 us (the panels come in no faster), so the grid stops at one.
// 256 x 256 tiles in parts were no faster on any of 18 products (sums of 256 KB: 15 us to meet), but for 2000 x 14336 x
// 4096 in two parts (105 against 120 us).  Measured before -> after, weights [K, N], bf16 out:
//   129 x 14336 x 4096  92 -> 35 us    512 x 14336 x 4096  95 -> 51    1024 x 14336 x 4096  94 -> 71
//   384 x 16384 x 1024  72 -> 24       512 x 8192 x 8192   57 -> 48     300 x 7168 x 7168   51 -> 40
#pragma once
#include "gemm_split.h"

namespace mi355q {

// The parts of a tile meet in pairs: parts 0 and 1, 2 and 3, then the sums of those pairs, and so on.  Of each pair the
// workgroup that comes second reads the first one's sums, adds them to its own and goes up (a + b = b + a, so the bits
// do not depend on who that is), by the ticket protocol of gemm_split.h; a sum without a partner goes up as it stands.
// Against adding all parts up in one place this needs no second copy of the sums in registers, and a workgroup reads
// log2(parts) sets of sums instead of parts - 1.  The sums of the subtree whose first leaf is p travel through the area
// of part p, which the subtree's own meetings are done with by then.
// NV values per thread, get(j) / set(j, v) with constant j.  Returns whether this workgroup holds the complete sums.
template <int NV, int THREADS, typename Get, typename Set>
__device__ __forceinline__ bool meet_in_pairs(const SplitArgs& s, int slot, int slots, int part, uint32_t* word, Get&& get, Set&& set) {
  constexpr int NW = NV / 2, CH = 8, NC = NW / CH;  // 8-byte words of a thread; words per step; steps
  static_assert(NW % CH == 0, "whole steps");
  const int64_t part_words = (int64_t)slots * NW * THREADS;
  unsigned long long* base = reinterpret_cast<unsigned long long*>(s.partials) + (int64_t)slot * NW * THREADS + threadIdx.x;
  for (int level = 0; ((s.parts - 1) >> level) > 0; ++level) {
    const int me = (part >> level) << level, other = ((part >> level) ^ 1) << level;
    if (other >= s.parts) continue;
    // one counter per pair: the pair is named by its right-hand part, which is the right-hand part of no other pair
    uint32_t* ticket = s.tickets + (slot * (s.parts - 1) + (me > other ? me : other) - 1) * kTicketStride;
    if (threadIdx.x == 0) *word = __hip_atomic_load(ticket, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    const bool other_in = *word != 0;  // then this workgroup is the second whatever happens, and its sums need not travel
    __syncthreads();
    if (!other_in) {
      unsigned long long* to = base + me * part_words;
      static_for<NW>([&](auto hc) {
        constexpr int h = decltype(hc)::value;
        const unsigned long long v = (unsigned long long)__float_as_uint(get(std::integral_constant<int, 2 * h>{})) |
                                     ((unsigned long long)__float_as_uint(get(std::integral_constant<int, 2 * h + 1>{})) << 32);
        __hip_atomic_store(to + h * THREADS, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if constexpr (h % CH == CH - 1) __builtin_amdgcn_sched_barrier(0);  // (all addresses at once do not fit the registers)
      });
      __builtin_amdgcn_s_waitcnt(0);  // the stores have been acknowledged before the ticket is drawn
      __syncthreads();
      if (threadIdx.x == 0) *word = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __syncthreads();
      if (*word == 0) return false;
      __syncthreads();  // the word has been read
    }
    if (threadIdx.x == 0) __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned long long* from = base + other * part_words;
    unsigned long long v[2][CH];
#pragma unroll
    for (int h = 0; h < CH; ++h) v[0][h] = __hip_atomic_load(from + h * THREADS, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    static_for<NC>([&](auto cc) {
      constexpr int c = decltype(cc)::value;
      if constexpr (c + 1 < NC) {
#pragma unroll
        for (int h = 0; h < CH; ++h)
          v[(c + 1) & 1][h] = __hip_atomic_load(from + ((c + 1) * CH + h) * THREADS, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      static_for<CH>([&](auto hc) {
        constexpr int j = 2 * (c * CH + decltype(hc)::value);
        const unsigned long long w = v[c & 1][decltype(hc)::value];
        set(std::integral_constant<int, j>{}, get(std::integral_constant<int, j>{}) + __uint_as_float((uint32_t)w));
        set(std::integral_constant<int, j + 1>{}, get(std::integral_constant<int, j + 1>{}) + __uint_as_float((uint32_t)(w >> 32)));
      });
      __builtin_amdgcn_sched_barrier(0);
    });
  }
  return true;
}

// A workgroup's tile and part of K.  Workgroups are dealt to the XCDs in turn; each XCD takes a contiguous range of
// (part, tile), the tiles of one part next to each other, so that the panels that its workgroups share come out of its L2.
// Parts are whole pairs of stages.
struct SplitPlace {
  int tile, tile_m, tile_n, part;
  template <bool A_KMAJOR, bool B_KMAJOR>
  __device__ __forceinline__ void find(GemmArgs& g, int parts) {
    const int bid = blockIdx.x, tiles = g.tiles_m * g.tiles_n, units = tiles * parts;
    const int xcd = bid & 7, per = units >> 3, rem = units & 7;
    const int unit = (xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per) + (bid >> 3);
    part = unit / tiles;
    tile = unit - part * tiles;
    tile_coords(tile, g.tiles_m, g.tiles_n, &tile_m, &tile_n);
    const int pairs = (g.K + 2 * kBK - 1) / (2 * kBK);
    const int k0 = (int)((int64_t)part * pairs / parts) * 2 * kBK, k1 = (int)((int64_t)(part + 1) * pairs / parts) * 2 * kBK;
    g.K = (g.K < k1 ? g.K : k1) - k0;
    g.A += (int64_t)k0 * (A_KMAJOR ? 1 : g.lda);
    g.B += (int64_t)k0 * (B_KMAJOR ? 1 : g.ldb);
  }
};

template <int BM, int BN, int WN, bool A_KMAJOR, bool B_KMAJOR, int FMT_A, int FMT_B>
__global__ __launch_bounds__(kWavesM * WN * 64) void fp8_gemm_tile_split_kernel(GemmArgs g, SplitArgs split) {
  constexpr int kThreads = kWavesM * WN * 64;
  constexpr int TM = BM / kWavesM, TN = BN / WN;
  constexpr int MT = TM / 32, NT = TN / 32;
  using Core = TileCore<BM, BN, WN, A_KMAJOR, B_KMAJOR, FMT_A, FMT_B>;
  static_assert(kWavesM * WN * epilogue_stage_floats<MT, NT>() * 4 <= Core::kRingBytes, "epilogue area overlays the ring");
  __shared__ __attribute__((aligned(1024))) uint8_t lds_ring[Core::kRingBytes];
  SplitPlace at;
  at.find<A_KMAJOR, B_KMAJOR>(g, split.parts);
  const int m0 = at.tile_m * BM, n0 = at.tile_n * BN;

  const int64_t batch = blockIdx.y;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = (wave / WN) * TM, wn = (wave % WN) * TN;
  Core core;
  core.init(g, lds_ring, wave, wm, wn);
  const int KT2 = ((g.K + kBK - 1) / kBK + 1) & ~1;
  core.set_lane_addresses(g);
  core.retarget(g, batch, m0, n0, true);
  core.template issue_stage<0>(0);
  core.template issue_stage<1>(1);
  core.first_fragments(false);
  auto k_step = [&](auto first_c, int kt) {
    const bool last = kt + 2 == KT2;
    if (last) core.retarget(g, batch, m0, n0, false);  // what the last pair loads arrives as zeros
    core.template k_pair<decltype(first_c)::value>(last ? -2 : kt, false, [] {});
  };
  k_step(std::true_type{}, 0);
  for (int kt = 2; kt < KT2; kt += 2) k_step(std::false_type{}, kt);

  // the ring is idle (the loads of the stages past K included) before the word and the epilogue overlay it
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  const int tiles = g.tiles_m * g.tiles_n;
  if (!meet_in_pairs<16 * MT * NT, kThreads>(
          split, (int)batch * tiles + at.tile, tiles * gridDim.y, at.part, reinterpret_cast<uint32_t*>(lds_ring),
          [&](auto jc) { constexpr int j = decltype(jc)::value; return core.acc[j / (16 * NT)][j / 16 % NT][j % 16]; },
          [&](auto jc, float v) { constexpr int j = decltype(jc)::value; core.acc[j / (16 * NT)][j / 16 % NT][j % 16] = v; }))
    return;
  __syncthreads();  // the word has been read
  float* stage = reinterpret_cast<float*>(lds_ring) + wave * epilogue_stage_floats<MT, NT>();
  if (g.fast_epi) epilogue_bf16_fast_any<MT, NT>(g, batch, core.acc, m0 + wm, n0 + wn, stage);
  else epilogue<MT, NT>(g, batch, core.acc, m0 + wm, n0 + wn, stage);
}

template <int BM, int BN, int WN, bool AK, bool BK_, int FA, int FB>
void launch_tile_split(const GemmArgs& g, const SplitArgs& split, int64_t batch, hipStream_t st) {
  GemmArgs a = g;
  a.tiles_m = (g.M + BM - 1) / BM;
  a.tiles_n = (g.N + BN - 1) / BN;
  dim3 grid((unsigned)(a.tiles_m * a.tiles_n * split.parts), (unsigned)batch);
  fp8_gemm_tile_split_kernel<BM, BN, WN, AK, BK_, FA, FB><<<grid, kWavesM * WN * 64, 0, st>>>(a, split);
}

}  // namespace mi355q
