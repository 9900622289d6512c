// fp8 GEMM for a handful of rows of A: instantiations of gemm_stream.h.
#include "gemm_stream.h"

namespace mi355q {

void launch_gemm_stream(const GemmArgs& g, int fmt_a, int fmt_b, const SplitPlan& p, const SplitArgs& split, int64_t batch, hipStream_t st) {
  if (fmt_a == MI355Q_E4M3FN && fmt_b == MI355Q_E4M3FN) launch_stream<MI355Q_E4M3FN, MI355Q_E4M3FN>(g, p, split, batch, st);
  else if (fmt_a == MI355Q_E4M3FN) launch_stream<MI355Q_E4M3FN, MI355Q_E5M2>(g, p, split, batch, st);
  else if (fmt_b == MI355Q_E4M3FN) launch_stream<MI355Q_E5M2, MI355Q_E4M3FN>(g, p, split, batch, st);
  else launch_stream<MI355Q_E5M2, MI355Q_E5M2>(g, p, split, batch, st);
}

}  // namespace mi355q
