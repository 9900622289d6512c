// The ring kernel for operands at any alignment: A K-major, B MN-major.
#include "gemm_dispatch.h"

namespace mi355q {
void launch_gemm_ragged_km(const GemmArgs& g, const SplitArgs& split, int fmt_a, int fmt_b, int64_t batch, hipStream_t st) {
  launch_ragged_by_format<false>(g, split, fmt_a, fmt_b, batch, st);
}
}  // namespace mi355q
