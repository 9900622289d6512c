// The meeting of workgroups that each hold one part of K of the same columns of C (split K): all in one place
// (split_exchange), or in pairs where the sums are large (meet_in_pairs).
//
// A workgroup stores its fp32 sums with device-scope atomic accesses, which go past the caches of its XCD to the level
// of memory that all XCDs share (no cache is written back or invalidated as a whole, which a fence would do), waits
// until they have been acknowledged, and draws a ticket; the workgroup that draws the last one adds the parts up in
// their order, whoever came last (the same bits from run to run), and goes on to the epilogue.  No workgroup ever
// waits for another.  The last one returns the counter to zero for the next launch.
//
// What it costs, measured on launches with and without it: 2 to 3 us (three dependent trips to that level of memory).
// The counters are a cache line apart: 256 workgroups drawing from counters that share lines serialised at that
// memory and took 2 us longer (16 parts of 16 strips).  The sums are laid out so that every access of a wave covers
// whole lines: with a thread's own eight columns in a row it was 4.4 instead of 2.2 us (two parts, 16 x 28672).
#pragma once
#include "gemm_tile.h"

namespace mi355q {

constexpr int kTicketStride = 16;                         // 32-bit words: one counter per 64-byte line
constexpr size_t kTicketBytes = MI355Q_FP8_GEMM_COUNTER_BYTES;  // the counters' area, in front of the sums, the same for every shape
constexpr int kMaxTickets = (int)(kTicketBytes / (kTicketStride * 4));

// The kernel of a product: 256 x 256 tiles (gemm_tile16.h, gemm_tile.h), rows of a ring tile (gemm_ring.h), or B streamed into
// registers (gemm_stream.h).
enum class GemmKind { kTile256, kRing16, kRing32, kRing64, kRing128, kRing192, kRing256, kStream };

struct SplitArgs {
  int parts;           // workgroups that share a strip or tile of C, one part of K each
  uint32_t* tickets;   // counters, zero between launches
  float* partials;
  GemmKind kind = GemmKind::kTile256;
};

// What a product runs on and how it is cut.
struct SplitPlan {
  GemmKind kind = GemmKind::kTile256;
  int nb = 0;                // columns per strip or tile
  int strips = 0, parts = 1;   // strips, or tiles
  int64_t tile_rows = 0;     // rows of sums a workgroup leaves in the workspace
  int64_t batch = 1;
  double stages_us = 0.0;    // ring kernel: what the stages of K are expected to take
  size_t workspace_bytes() const {
    return parts < 2 ? 0 : kTicketBytes + (size_t)parts * strips * batch * tile_rows * nb * sizeof(float);
  }
};
SplitPlan split_plan(bool a_kmajor, int64_t lda, bool b_kmajor, int64_t ldb, int64_t M, int64_t N, int64_t K, int64_t batch, bool may_split,
                     bool fp32_rows = false,   // fp32 results that ring_epilogue_rows writes
                     bool ring_only = false);  // the ring kernel's forms alone

// The counter, looked at ahead of time (before waits that the workgroup has anyway): parts - 1 means that every other
// part has arrived; then this workgroup is the last whatever happens, and its own sums need not travel.
__device__ __forceinline__ uint32_t split_look(const SplitArgs& s, int slot) {
  return __hip_atomic_load(s.tickets + slot * kTicketStride, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// NV values per thread, get(j) / set(j, v) with constant j; `mine`: the thread holds values that matter.
// Returns whether this workgroup goes on to the epilogue (with the complete sums set).
template <int NV, int THREADS, typename Get, typename Set>
__device__ __forceinline__ bool split_exchange(const SplitArgs& s, int slot, int slots, int part, bool mine, bool others_in,
                                               uint32_t* word, Get&& get, Set&& set) {
  constexpr int NW = NV / 2;
  const int64_t part_words = (int64_t)slots * NW * THREADS;
  unsigned long long* base = reinterpret_cast<unsigned long long*>(s.partials) + (int64_t)slot * NW * THREADS + threadIdx.x;
  if (!others_in) {
    if (mine) {
      unsigned long long* to = base + part * part_words;
#pragma unroll
      for (int h = 0; h < NW; ++h) {
        const unsigned long long v = (unsigned long long)__float_as_uint(get(2 * h)) | ((unsigned long long)__float_as_uint(get(2 * h + 1)) << 32);
        __hip_atomic_store(to + h * THREADS, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    __builtin_amdgcn_s_waitcnt(0);  // the stores have been acknowledged before the ticket is drawn
    __syncthreads();
    if (threadIdx.x == 0) *word = __hip_atomic_fetch_add(s.tickets + slot * kTicketStride, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (*word != (uint32_t)s.parts - 1) return false;
  }
  if (threadIdx.x == 0) __hip_atomic_store(s.tickets + slot * kTicketStride, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (!mine) return true;
  float own[NV];
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    own[j] = get(j);
    set(j, 0.0f);
  }
  constexpr int kAhead = NW <= 8 ? 4 : (NW <= 16 ? 2 : 1);  // parts whose loads are in flight together
  for (int p = 0; p < s.parts; p += kAhead) {
    unsigned long long v[kAhead][NW];
#pragma unroll
    for (int q = 0; q < kAhead; ++q) {
      const int pq = p + q < s.parts ? p + q : s.parts - 1;
#pragma unroll
      for (int h = 0; h < NW; ++h) v[q][h] = __hip_atomic_load(base + pq * part_words + h * THREADS, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
#pragma unroll
    for (int q = 0; q < kAhead; ++q) {
      if (p + q < s.parts) {
        const bool me = p + q == part;
#pragma unroll
        for (int h = 0; h < NW; ++h) {
          set(2 * h, get(2 * h) + (me ? own[2 * h] : __uint_as_float((uint32_t)v[q][h])));
          set(2 * h + 1, get(2 * h + 1) + (me ? own[2 * h + 1] : __uint_as_float((uint32_t)(v[q][h] >> 32))));
        }
      }
    }
  }
  return true;
}

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
    if (__builtin_expect(!other_in, true)) {
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

}  // namespace mi355q
