// GEMM dispatch for gfx950 (MI355X): the launch of the MFMA kernels
// (gemm_w4.h: 256x256 tiles; gemm_128.h: 128x128 tiles; gemm_any.h: operands
// of any alignment), all of which take every storage order of A and B, as
// the launch planner (launch_plan.h) decides.
//
// Semantics follow frisk.gemm (include/Dialect/Frisk/IR/FriskOps.td:252-292):
// C = op(A).op(B) when clear_accum, else C += op(A).op(B).
//
#include <algorithm>

#include "common.h"

#include "gemm_common.h"
#include "kernels.h"

namespace frisk {

namespace {

// One storage order: AM = A stored [K, M] (trans_a), BM = B stored [K, N]
// (not trans_b).
template <bool AM, bool BM>
hipError_t run_layout(const GemmArgs& g, hipStream_t s, const MfmaChoice& c, void* ws) {
  if (c.slices > 1) {
    if (c.big) return gemm_w4_split_layout<AM, BM>(g, c.slices, c.kb_slice, ws, s);
    return gemm_128_split_layout<AM, BM>(g, c.slices, c.kb_slice, ws, s);
  }
  if (c.big) return gemm_w4_layout<AM, BM>(g, s);
  // A requested 2x2 grid runs as the library's own 128x128 launch (its
  // stage depth); the other grids run 64-byte stages.
  if (g.tile == 128 && !(g.wave_m == 2 && g.wave_n == 2)) return gemm_128_grid_layout<AM, BM>(g, s);
  return gemm_128_layout<AM, BM>(g, s);
}

}  // namespace

// The launch follows plan::mfma_choice (launch_plan.h): the library's own
// choice, or the requested variant with the K slices it names.
hipError_t gemm_mfma(const GemmArgs& g, hipStream_t s, void* workspace, int64_t workspace_bytes) {
  const int cus = device_cus();
  const int64_t need = plan::workspace_bytes(shape_of(g), plan::Route::Mfma, cus);
  const bool ws = workspace && need > 0 && workspace_bytes >= need;
  const MfmaChoice c = gemm_mfma_choice(g, cus, ws);
  void* tree_ws = c.slices > 1 ? workspace : nullptr;
  switch ((g.trans_a ? 2 : 0) | (g.trans_b ? 0 : 1)) {
    case 0: return run_layout<false, false>(g, s, c, tree_ws);  // A [M,K], B [N,K]
    case 1: return run_layout<false, true>(g, s, c, tree_ws);   // A [M,K], B [K,N]
    case 2: return run_layout<true, false>(g, s, c, tree_ws);   // A [K,M], B [N,K]
    default: return run_layout<true, true>(g, s, c, tree_ws);   // A [K,M], B [K,N]
  }
}

hipError_t gemm_any(const GemmArgs& g, hipStream_t s, void* workspace, int64_t workspace_bytes) {
  plan::SplitPlan p = plan::any_plan(shape_of(g), device_cus(), true);
  if (!workspace || workspace_bytes < p.workspace_bytes)
    p = plan::any_plan(shape_of(g), device_cus(), false);
  hipError_t e;
  switch ((g.trans_a ? 2 : 0) | (g.trans_b ? 0 : 1)) {
    case 0: e = gemm_any_layout<false, false>(g, p, workspace, s); break;
    case 1: e = gemm_any_layout<false, true>(g, p, workspace, s); break;
    case 2: e = gemm_any_layout<true, false>(g, p, workspace, s); break;
    default: e = gemm_any_layout<true, true>(g, p, workspace, s);
  }
  if (e != hipSuccess || p.slices <= 1) return e;
  return gemm_splitk_sum(workspace, p.slices, plan::any_partial_pitch(g.n), g, s);
}

}  // namespace frisk
