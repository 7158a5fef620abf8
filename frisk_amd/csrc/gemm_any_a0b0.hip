// The any-alignment MFMA GEMM (gemm_any.h) for trans_a = 0, trans_b = 0:
// A stored [M, K], B stored [K, N].
#include "gemm_any.h"

namespace frisk {
template hipError_t gemm_any_layout<false, true>(const GemmArgs&, const plan::SplitPlan&, void*,
                                             hipStream_t);
}  // namespace frisk
