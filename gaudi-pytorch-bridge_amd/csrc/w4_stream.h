// The stream kernel of the 4-bit products (w4_stream.hip): which problems it takes, how it cuts them, its launch.
#pragma once
#include "w4_common.h"

namespace mi355q {

constexpr int kW4StBN = 512;                     // columns of a workgroup
constexpr int kW4StRows = 16;
constexpr int kW4StMostParts = 16;
constexpr int64_t kW4StMostPitch = 1LL << 22;    // elements of A, words of the weights: 16 and 128 rows of them are 31-bit offsets
constexpr int kW4Bf16 = -1;                      // in the place of an fp8 format: bf16 activations

// parts 0: the kernel does not take the problem.
struct W4StreamPlan {
  int strips = 0, parts = 0;
  size_t workspace_bytes() const {
    return parts < 2 ? 0 : kW4TicketBytes + (size_t)parts * strips * kW4StRows * kW4StBN * sizeof(float);
  }
};
W4StreamPlan w4_stream_plan(int64_t M, int64_t N, int64_t K, int64_t group, int scale_f32, bool a16);

// act: MI355Q_E4M3FN, MI355Q_E5M2 or kW4Bf16; workspace: as w4_stream_plan wants it; last_alone: the part that arrives last adds
// all of them up (what happens to the shares of parts that see nobody arrive in time).
void launch_w4_stream(W4Args a, int act, const W4StreamPlan& plan, void* workspace, bool last_alone, hipStream_t st);

}  // namespace mi355q
