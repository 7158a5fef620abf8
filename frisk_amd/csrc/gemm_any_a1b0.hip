// The any-alignment MFMA GEMM (gemm_any.h) for trans_a = 1, trans_b = 0:
// A stored [K, M], B stored [K, N].
#include "gemm_any.h"

namespace frisk {
template hipError_t gemm_any_layout<true, true>(const GemmArgs&, const plan::SplitPlan&, void*,
                                             hipStream_t);
}  // namespace frisk
