// Packed 4-bit weights (groups of 128, bf16 scales) against at most 16 rows of fp8 or bf16 activations.
//
// Such a product is bound by reading the packed words once.  A workgroup owns 512 columns and one part of K: 256-byte pieces of such
// a matrix stream at 5.9 to 6.3 TB/s, 128-byte ones (the strips of w4a8_wide_kernel) at 5.1 to 5.5 (117 MB, reads alone: 18.7 to
// 19.9 against 21.3 to 22.9 us).  Eight waves multiply, 64 columns each, and four load: a compute unit keeps about 32 KB of lines on
// their way and a wave that asks for more stalls in the issue, with whatever it still had to multiply (eight waves that did both,
// each on a stream of its own: 29.3 us at 16 x 8192 x 28672, where the loads alone took 20).  A stage is a group of 128 k, one barrier each.
//
// The product runs in bf16, for fp8 activations too: v_cvt_scalef32_pk_bf16_fp8 makes the nibbles, which are e4m3 codes of q x 2^-9, and
// the activations bf16, exactly.  At 16 rows the matrix unit has room for its lower rate, the launch that splits bf16 activations
// into fp8 planes (3 to 4 us) goes, and so does the fp8 forms' rounding inside a product: over the shapes above and uint4 and int4
// weights, fp32 results are 1e-7 from the exact ones (2-norm) where the 16x16x128 f8f6f4 form of w4a8_wide_kernel gives 1e-5 to
// 5e-5 and 16x16x32 in fp8 2e-4 to 5e-4.
//
// The parts of K meet in the workspace.  The sums of 512 columns are 32 KiB a part: one workgroup that reads four of them takes 3 us for
// that alone.  So each part adds up its share of the columns, if it sees the others arrive within a few looks; the one that
// arrives last also takes the shares of those that gave up.  Nobody waits longer than those looks.  (16 x 8192 x 28672 28.0 -> 26.7 us,
// 16 x 14336 x 4096 in eight parts 18.6 -> 18.0.)
//
// Against w4a8_wide_kernel, us, weights cold: bf16 activations 16 x 8192 x 28672 33.3 -> 27.4, 16 x 14336 x 4096 22.7 -> 15.9, 8 x 4096 x
// 4096 15.6 -> 10.2; fp8 29.7 -> 26.5, 19.5 -> 14.8, 13.2 -> 10.0.  What is left of the 27: 20 of loads, 3 for the parts' meeting, and the
// first stage's way in and the last one's through the multiplying waves.
#include <algorithm>

#include "w4_stream.h"

namespace mi355q {

constexpr int kW4StConsumers = 8, kW4StLoaders = 4;
constexpr int kW4StThreads = (kW4StConsumers + kW4StLoaders) * 64;
constexpr int kW4StTiles = 4;                                  // column tiles of 16 of a consumer
constexpr int kW4StUnits = kW4StConsumers * kW4StTiles;        // tiles of a workgroup: what the parts deal out
constexpr int kW4StWeights = kBK * kW4StBN / 2;                // bytes of a stage's weights
constexpr int kW4StScale = kW4StBN * 2, kW4StZp = kW4StBN / 2;
constexpr int w4_stream_stage(bool a16) { return kW4StWeights + kW4StRows * kBK * (a16 ? 2 : 1) + kW4StScale + kW4StZp; }
constexpr int kW4StStages = 3;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// Eight k of one operand of v_mfma_f32_16x16x32_bf16.  Weights are q x 2^-kW4StShift, with which the sums of a group stay inside fp32
// whatever the activations, and with denormal ones too every product is still a multiple of fp32's smallest value; sums of activations
// alone are taken with ones of the same size.  The sums over the groups are in the results' own units: at 2^-kW4StShift of them
// results below 2^-113 lost bits (rows of 2^-120 under scales of 2^-27 all of them).
// fp8 activations need none of that: their sums of a group are below 2^27.
constexpr int kW4StShift = 12;
constexpr int w4_st_shift(int act) { return act == kW4Bf16 ? kW4StShift : 0; }
template <int ACT>
__device__ __forceinline__ u32x4 w4_st_weights(uint32_t w) {  // eight nibbles, the even ones for k 0 .. 3
  const int even = (int)(w & 0x0f0f0f0fu), odd = (int)((w >> 4) & 0x0f0f0f0fu);
  constexpr float s = 512.0f / (float)(1 << w4_st_shift(ACT));  // 2^9 for the code
  return u32x4{__builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(even, s, false)),
               __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(even, s, true)),
               __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(odd, s, false)),
               __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(odd, s, true))};
}
template <int ACT>
__device__ __forceinline__ u32x4 w4_st_ones() {
  constexpr uint32_t one = (uint32_t)(127 - w4_st_shift(ACT)) << 7, two = one << 16 | one;
  return u32x4{two, two, two, two};
}
template <int ACT>
__device__ __forceinline__ u32x4 w4_st_widen(uint32_t lo, uint32_t hi) {  // eight fp8 activations
  const auto two = [](uint32_t v, auto hc) {
    constexpr bool high = decltype(hc)::value;
    if constexpr (ACT == MI355Q_E4M3FN) return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((int)v, 1.0f, high));
    else return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_bf8((int)v, 1.0f, high));
  };
  return u32x4{two(lo, std::false_type{}), two(lo, std::true_type{}), two(hi, std::false_type{}), two(hi, std::true_type{})};
}
__device__ __forceinline__ f32x4 w4_st_mfma(const u32x4& w, const u32x4& a, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w), __builtin_bit_cast(bf16x8, a), c, 0, 0, 0);
}

// A strip's word in the workspace, zero between launches: parts arrived (bits 0 - 7), shares taken (bit 8 + part), parts that have
// seen all arrive (bits 24 up).  A part arrives with its share taken and may give it back only while others are missing, so the
// last one knows at once which shares are left to it.  Whoever is the last to have seen all arrive returns the word to zero.
constexpr uint32_t w4_arrival(int part) { return 1u + (256u << part); }
constexpr uint32_t kW4AllSeen = 1u << 24;
constexpr int kW4Looks = 12;  // about 0.7 us each

template <int ACT, bool HAS_Z>
__global__ __launch_bounds__(kW4StThreads, 1) void w4_stream_kernel(W4Args a, int looks) {
  constexpr bool A16 = ACT == kW4Bf16;
  constexpr int kActBytes = A16 ? 2 : 1, kARow = kBK * kActBytes;
  constexpr int S = kW4StStages, kStage = w4_stream_stage(A16);
  constexpr int kOffA = kW4StWeights, kOffScale = kOffA + kW4StRows * kARow, kOffZp = kOffScale + kW4StScale;
  static_assert(kStage % 256 == 0, "rows of weights stay aligned");
  static_assert(S == 3, "the loaders' waits are for one stage behind the one they wait for");
  __shared__ __attribute__((aligned(1024))) uint8_t lds[S * kStage];
  __shared__ __attribute__((aligned(16))) float scales[2][kW4StBN], zeros[2][HAS_Z ? kW4StBN : 4];  // zeros: minus the zero-points
  __shared__ uint32_t word, again;

  const GemmArgs& g = a.g;
  const int strips = (g.N + kW4StBN - 1) / kW4StBN;
  const int strip = blockIdx.x % strips, part = blockIdx.x / strips;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, r16 = lane & 15, gk = lane >> 4;
  const int n0 = strip * kW4StBN;
  const int groups = g.K / kBK;
  const int g0 = (int)((int64_t)part * groups / a.ksplit), KT = (int)((int64_t)(part + 1) * groups / a.ksplit) - g0;
  f32x4 total[kW4StTiles];
#pragma unroll
  for (int t = 0; t < kW4StTiles; ++t) total[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  // bf16 activations near the end of fp32's range: where a sum may not be finite the workgroup walks its part once more, at
  // 2^-kW4StShift of the size, for the sums that are not.  The question costs 0.2 us of 12 to 28; both sums side by side 0.3 to 1.2.
  bool second = false;
  const auto once_more = [&] {
    if (!A16 || second) return false;
    second = __builtin_amdgcn_readfirstlane((int)again) != 0;
    return second;
  };
  if (A16 && threadIdx.x == 0) again = 0;  // (in front of the barrier of the first stage)

  if (wave >= kW4StConsumers) {
    const int wq = wave - kW4StConsumers;
    constexpr int kNowhere = 0x7fffffff;  // an offset that no descriptor covers: reads as zero
    const int ld = (int)a.ld_packed;
    // Weights: four rows of sixteen 16-byte slots per load, loader wq rows 32 wq .. 32 wq + 31; slot s of row r sits in LDS at slot
    // s ^ (r % 16), which keeps the 16 rows of a transposing read off each other's banks.  (The first slot of a row is always
    // inside N: every load goes to memory, which the counted waits rely on.)
    int vo_w[4], step_w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int slot = r16 ^ (4 * j + gk);
      const bool inside = n0 + 32 * slot < g.N;
      vo_w[j] = inside ? (32 * wq + 4 * j + gk) * ld + slot * 16 : kNowhere;
      step_w[j] = inside ? 16 * ld : 0;
    }
    // Activations: rows past M read the last one.  bf16: four rows of 256 bytes per load, one load each; fp8: eight rows of 128,
    // by loaders 0 and 1.  Scales by loader 0 (fp8: 2), zero-points by the next; the others repeat one of these, so that all have
    // the same number of loads on their way.
    constexpr int kSlots = kARow / 16, kARows = 64 / kSlots, kALoads = kW4StRows / kARows;
    const int a_load = wq % kALoads, a_row = a_load * kARows + lane / kSlots;
    const int a_slot = (lane % kSlots) ^ (A16 ? a_row : (a_row >> 1) & 7);
    const int vo_a = (a_row < g.M ? a_row : g.M - 1) * (int)(g.lda * kActBytes) + a_slot * 16;
    const bool bring_zp = HAS_Z && a.zp != nullptr && (wq & 1) != 0;
    const int vo_row = bring_zp ? (n0 + 8 * lane < g.N ? lane * 4 : kNowhere) : (n0 + 8 * lane < g.N ? lane * 16 : kNowhere);
    const uint8_t* row_from = bring_zp ? a.zp + n0 / 2 : a.scale + n0 * 2;
    const int64_t row_step = bring_zp ? g.N / 2 : (int64_t)g.N * 2;
    const int row_at = bring_zp ? kOffZp : kOffScale;
    constexpr int kOps = 8 + 2;
    static_assert((S - 1) * kOps <= 63, "vmcnt holds 6 bits");
    const auto view = [](const uint8_t* p) {
      const uint64_t b = reinterpret_cast<uint64_t>(p);
      return i32x4{__builtin_amdgcn_readfirstlane((int)(uint32_t)b), __builtin_amdgcn_readfirstlane((int)(uint32_t)((b >> 32) & 0xffffu)), 0x7ffffff0, 0x00020000};
    };
    const uint32_t base = (uint32_t)(uintptr_t)(LDS_AS uint8_t*)lds;
    auto issue = [&](int off, int kt) {
      const int64_t group = g0 + kt;
      const i32x4 rw = view(a.packed + group * kBK * a.ld_packed + n0 / 2);
#pragma unroll
      for (int j = 0; j < 8; ++j) w4_dma16<true>(rw, vo_w[j & 3] + (j >> 2) * step_w[j & 3], base + off + (8 * wq + j) * 1024);
      w4_dma16(view(g.A + group * kARow), vo_a, base + off + kOffA + a_load * 1024);
      if (bring_zp) w4_dma4(view(row_from + group * row_step), vo_row, base + off + row_at);
      else w4_dma16(view(row_from + group * row_step), vo_row, base + off + row_at);
    };
    // the scales of a stage and minus its zero-points as fp32, two columns per lane, for the fold one stage later
    const uint32_t flip = a.is_signed ? 0x88u : 0u;
    auto rows = [&](int off, int slot) {
      const int n = (wq * 64 + lane) * 2;
      const uint32_t s2 = *reinterpret_cast<const uint32_t*>(lds + off + kOffScale + 2 * n);
      f32x2 s = {__uint_as_float(s2 << 16), __uint_as_float(s2 & 0xffff0000u)};
      if constexpr (A16) {
        if (!second) {
          s *= (float)(1 << kW4StShift);
          if (!(__builtin_fabsf(s[0]) < __builtin_inff() && __builtin_fabsf(s[1]) < __builtin_inff())) again = 1;  // scales from 2^116 on
        }
      }
      *reinterpret_cast<f32x2*>(&scales[slot][n]) = s;
      if constexpr (HAS_Z) {
        const uint32_t z2 = (a.zp != nullptr ? lds[off + kOffZp + n / 2] : 0u) ^ flip;
        *reinterpret_cast<f32x2*>(&zeros[slot][n]) = f32x2{-(float)(z2 & 15u), -(float)(z2 >> 4)};
      }
    };
    do {
#pragma unroll
      for (int s = 0; s < S - 1; ++s)
        if (s < KT) issue(s * kStage, s);
      int wr_off = (S - 1) * kStage, rd_off = 0;
      for (int kt = 0; kt < KT; ++kt) {
        // stage kt has landed when only the loads of those after it are on their way
        constexpr int c = (S - 2) * kOps;
        if (kt + S - 2 < KT) __builtin_amdgcn_s_waitcnt((c & 15) | ((c >> 4) << 14) | 0x0f70);
        else __builtin_amdgcn_s_waitcnt(0x0f70);
        __syncthreads();  // stage kt is in LDS for the consumers, who are done with stage kt - 1
        if (kt + S - 1 < KT) issue(wr_off, kt + S - 1);
        rows(rd_off, kt & 1);
        wr_off = wr_off + kStage == S * kStage ? 0 : wr_off + kStage;
        rd_off = rd_off + kStage == S * kStage ? 0 : rd_off + kStage;
      }
      __syncthreads();  // the consumers' fold of the last stage
    } while (once_more());
  } else {
    const uint32_t flip = a.is_signed ? 0x88888888u : 0u;  // signed nibble s = (q ^ 8) - 8
    // lane: row m = lane % 16 of A; columns n0 + 64 wave + 16 t + 4 gk + e.  The transposing read of step pair p points at k-row
    // 64 p + 16 gk + w4_nibble_row(lane % 16); the lane's k are 64 p + 16 gk .. + 15 then, in two steps.
    int woff[2];  // of tile 0 and of tile 2; tile t + 1: 8 bytes on
    const int krow = 16 * gk + w4_nibble_row(r16);
#pragma unroll
    for (int s = 0; s < 2; ++s) woff[s] = krow * 256 + (((2 * wave + s) ^ (krow & 15)) << 4);
    int aoff[2][A16 ? 2 : 1];
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int i = 0; i < (A16 ? 2 : 1); ++i)
        aoff[p][i] = kOffA + r16 * kARow + (A16 ? (8 * p + 2 * gk + i) ^ r16 : (4 * p + gk) ^ ((r16 >> 1) & 7)) * 16;
    const int col = 64 * wave + 4 * gk;
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 acc[2][kW4StTiles];
    float sums[2] = {0.0f, 0.0f};
    int rd_off = 0;
    auto fold = [&](auto bc) {
      constexpr int B = decltype(bc)::value;
#pragma unroll
      for (int t = 0; t < kW4StTiles; ++t) {
        const f32x4 s = *reinterpret_cast<const f32x4*>(&scales[B][col + 16 * t]);
        f32x4 d = acc[B][t];  // the zero-points first, so that what cancels does so here
        if constexpr (HAS_Z) {
          const f32x4 z = *reinterpret_cast<const f32x4*>(&zeros[B][col + 16 * t]);
#pragma unroll
          for (int e = 0; e < 4; ++e) d[e] = __builtin_fmaf(z[e], sums[B], d[e]);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) total[t][e] = __builtin_fmaf(d[e], s[e], total[t][e]);
      }
    };
    auto stage = [&](auto bc, auto hpc) {
      constexpr int B = decltype(bc)::value;
      __syncthreads();  // the stage is in LDS, and so are the fp32 rows of the one before
      const uint8_t* st = lds + rd_off;
      i32x2 w[2][kW4StTiles];
      u32x4 act[2][2];
#pragma unroll
      for (int p = 0; p < 2; ++p) {
#pragma unroll
        for (int t = 0; t < kW4StTiles; ++t)
          w[p][t] = __builtin_amdgcn_ds_read_tr4_b64_v2i32((LDS_AS i32x2*)((LDS_AS uint8_t*)st + woff[t >> 1] + (t & 1) * 8 + p * 64 * 256));
        const u32x4 lo = *reinterpret_cast<const u32x4*>(st + aoff[p][0]);
        if constexpr (A16) {
          act[p][0] = lo;
          act[p][1] = *reinterpret_cast<const u32x4*>(st + aoff[p][A16 ? 1 : 0]);
        } else {
          act[p][0] = lo;
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (!A16) {
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          const u32x4 v = act[p][0];
          act[p][0] = w4_st_widen<ACT>(v[0], v[1]);
          act[p][1] = w4_st_widen<ACT>(v[2], v[3]);
        }
      }
      f32x4 rs = zero;
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          if constexpr (HAS_Z) rs = w4_st_mfma(w4_st_ones<ACT>(), act[p][h], rs);
#pragma unroll
          for (int t = 0; t < kW4StTiles; ++t) acc[B][t] = w4_st_mfma(w4_st_weights<ACT>((uint32_t)w[p][t][h] ^ flip), act[p][h], p == 0 && h == 0 ? zero : acc[B][t]);
        }
      // the stage before this one, whose MFMAs finished long ago, behind those just issued
      if constexpr (decltype(hpc)::value) fold(std::integral_constant<int, 1 - B>{});
      sums[B] = rs[0];
      rd_off = rd_off + kStage == S * kStage ? 0 : rd_off + kStage;
    };
    using T = std::true_type;
    using F = std::false_type;
    // Before the barrier of the last stage's rows: whether the sums of the stages before it are finite.  (The last fold rounds once: it
    // leaves an infinity only where the part's sum is one.)
    const auto in_range = [&] {
      f32x4 v = zero;  // or NaN
#pragma unroll
      for (int t = 0; t < kW4StTiles; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = __builtin_fmaf(total[t][e], 0.0f, v[e]);
      if (!((v[0] + v[1]) + (v[2] + v[3]) == 0.0f)) again = 1;
    };
    f32x4 first[A16 ? kW4StTiles : 1];
    do {
      if (second) {
        rd_off = 0;
#pragma unroll
        for (int t = 0; t < kW4StTiles; ++t) {
          first[A16 ? t : 0] = total[t];
          total[t] = zero;
        }
      }
      stage(std::integral_constant<int, 0>{}, F{});
      int kt = 1;
      for (; kt + 1 < KT; kt += 2) {
        stage(std::integral_constant<int, 1>{}, T{});
        stage(std::integral_constant<int, 0>{}, T{});
      }
      if (kt < KT) stage(std::integral_constant<int, 1>{}, T{});
      if constexpr (A16) in_range();
      __syncthreads();  // the fp32 rows of the last stage
      if (KT & 1) fold(std::integral_constant<int, 0>{});
      else fold(std::integral_constant<int, 1>{});
    } while (once_more());
    if (second) {
#pragma unroll
      for (int t = 0; t < kW4StTiles; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float v = first[A16 ? t : 0][e];
          total[t][e] = __builtin_isfinite(v) ? v : total[t][e] * (float)(1 << kW4StShift);
        }
    }
  }

  const ScalarScales scalars = load_scalar_scales(g);
  const float sa = w4_row_scale(g, scalars, r16);
  const auto finish = [&](int unit, const f32x4& sum) {
    const int n = n0 + 16 * unit + 4 * gk;
    w4_store4(g, r16, n, sum, sa, w4_bias4(g, n));
  };
  if (a.ksplit == 1) {
    if (wave >= kW4StConsumers) return;
#pragma unroll
    for (int t = 0; t < kW4StTiles; ++t) finish(wave * kW4StTiles + t, total[t]);
    return;
  }

  // Sums travel as 8-byte words: [part][strip][unit][half][lane], rows past M not at all.
  const int64_t part_words = (int64_t)strips * kW4StUnits * 128;
  unsigned long long* const sums = reinterpret_cast<unsigned long long*>(a.partials) + (int64_t)strip * kW4StUnits * 128 + lane;
  uint32_t* const at = a.tickets + strip * a.ticket_stride;
  if (wave < kW4StConsumers) {
    if (r16 < g.M) {
#pragma unroll
      for (int t = 0; t < kW4StTiles; ++t)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          __hip_atomic_store(sums + part * part_words + ((wave * kW4StTiles + t) * 2 + h) * 64,
                             (unsigned long long)__float_as_uint(total[t][2 * h]) | ((unsigned long long)__float_as_uint(total[t][2 * h + 1]) << 32),
                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __builtin_amdgcn_s_waitcnt(0);  // acknowledged before the part arrives
  }
  __syncthreads();
  // the shares this workgroup takes, one bit each
  if (threadIdx.x == 0) {
    const uint32_t parts = (uint32_t)a.ksplit, all = (1u << a.ksplit) - 1u;
    uint32_t v = __hip_atomic_fetch_add(at, w4_arrival(part), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + w4_arrival(part);
    uint32_t take = 1u << part;
    if ((v & 255u) == parts) {
      take |= all & ~(v >> 8);
    } else {
      for (int i = 0; i < looks && (v & 255u) != parts; ++i) {
        __builtin_amdgcn_s_sleep(1);
        v = __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      while ((v & 255u) != parts) {  // give the share back, unless the last one arrives at this moment (at most `parts` others change the word)
        if (__hip_atomic_compare_exchange_strong(at, &v, v & ~(256u << part), __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
          take = 0;
          break;
        }
      }
    }
    word = take;
  }
  __syncthreads();
  uint32_t take = word;
  if (take == 0) return;
  if (threadIdx.x == 0) {
    const uint32_t v = __hip_atomic_fetch_add(at, kW4AllSeen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + kW4AllSeen;
    // (a bit is left for every part that goes on; those that gave up have none)
    if ((int)(v >> 24) == __builtin_popcount((v >> 8) & 0xffffu)) __hip_atomic_store(at, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (wave >= kW4StConsumers) return;
  for (; take != 0; take &= take - 1) {
    const int share = __builtin_ctz(take);
    for (int unit = share + a.ksplit * wave; unit < kW4StUnits; unit += a.ksplit * kW4StConsumers) {
      f32x4 sum = {0.f, 0.f, 0.f, 0.f};
      constexpr int kAhead = 4;  // parts whose loads are in flight together
      for (int p = 0; p < a.ksplit; p += kAhead) {
        unsigned long long v[kAhead][2];
        if (r16 < g.M) {
#pragma unroll
          for (int q = 0; q < kAhead; ++q)
#pragma unroll
            for (int h = 0; h < 2; ++h)
              v[q][h] = __hip_atomic_load(sums + (p + q < a.ksplit ? p + q : p) * part_words + (unit * 2 + h) * 64, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
          for (int q = 0; q < kAhead; ++q)
            if (p + q < a.ksplit) {
#pragma unroll
              for (int h = 0; h < 2; ++h) {
                sum[2 * h] += __uint_as_float((uint32_t)v[q][h]);
                sum[2 * h + 1] += __uint_as_float((uint32_t)(v[q][h] >> 32));
              }
            }
        }
      }
      finish(unit, sum);
    }
  }
}

// At most 16 rows (a second row tile would double the products of a stage, which take nearly as long as its loads).  The parts are those
// expected to take least: a stage takes 1 us (40 KB/us, what a compute unit takes in), or its share of 5.8 TB/s
// where more than 160 workgroups run, their meeting 2.9 and a part 0.15 (us, bf16 activations,
// in 1 / 2 / 4 / 8 / 16 parts: 8 x 4096 x 4096 36.0 / 22.9 / 14.5 / 11.1 / 10.2, 16 x 14336 x 4096 114 / 62 / 34.3 / 21.3 / 15.6; fp8, 3 x 3200 x
// 12736 in 4 / 6 / 10 14.5 / 13.7 / 14.2).  Without room for the parts, K in one: w4a8_wide_kernel's strips are half as wide and
// fill the chip better then, so the caller goes there where the plan wants parts.  So do short products on fp8 activations, which the
// narrower strips serve with fewer parts or none: 16 x 768 x 28672 10.0 there and 10.5 here, 16 x 1024 x 40000 13.1 and 14.9, but 16 x
// 1024 x 28672 11.2 and 10.9, 4 x 1024 x 1024 9.5 and 8.2 (bf16 activations have their split to save: 16 x 768 x 28672 12.7 and 10.5).
W4StreamPlan w4_stream_plan(int64_t M, int64_t N, int64_t K, int64_t group, int scale_f32, bool a16) {
  W4StreamPlan p;
  if (group != kBK || scale_f32 || M < 1 || M > kW4StRows || N <= 0 || K <= 0 || N > (1LL << 24) || K > (1LL << 24)) return p;
  p.strips = (int)((N + kW4StBN - 1) / kW4StBN);
  if (!a16 && K < (p.strips <= 64 ? 1024 : 2048)) return p;
  const int groups = (int)(K / kBK), most = std::min({256 / p.strips, groups / 2, kW4StMostParts});
  double best = 0.0;
  for (int n = 1; n <= std::max(most, 1); ++n) {
    const double us = (double)((groups + n - 1) / n) * std::max(1.0, 0.0062 * (double)(n * p.strips)) + (n > 1 ? 2.9 + 0.15 * (double)n : 0.0);
    if (n > 1 && us >= best) continue;
    best = us;
    p.parts = n;
  }
  return p;
}

void launch_w4_stream(W4Args a, int act, const W4StreamPlan& plan, void* workspace, bool last_alone, hipStream_t st) {
  a.ksplit = plan.parts;
  if (plan.parts > 1) {
    a.tickets = static_cast<uint32_t*>(workspace);
    a.partials = reinterpret_cast<float*>(static_cast<uint8_t*>(workspace) + kW4TicketBytes);
    // the counters as far apart as their area allows
    a.ticket_stride = 16;
    while ((size_t)plan.strips * a.ticket_stride * 4 > kW4TicketBytes) a.ticket_stride /= 2;
  }
  const unsigned grid = (unsigned)(plan.strips * plan.parts);
  const auto launch = [&](auto actc) {
    constexpr int ACT = decltype(actc)::value;
    if (a.zp != nullptr || a.is_signed) w4_stream_kernel<ACT, true><<<grid, kW4StThreads, 0, st>>>(a, last_alone ? 0 : kW4Looks);
    else w4_stream_kernel<ACT, false><<<grid, kW4StThreads, 0, st>>>(a, last_alone ? 0 : kW4Looks);
  };
  if (act == kW4Bf16) launch(std::integral_constant<int, kW4Bf16>{});
  else if (act == MI355Q_E4M3FN) launch(std::integral_constant<int, MI355Q_E4M3FN>{});
  else launch(std::integral_constant<int, MI355Q_E5M2>{});
}

}  // namespace mi355q
