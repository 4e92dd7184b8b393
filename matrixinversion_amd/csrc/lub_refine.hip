// lub_refine.hip -- entry points of the refined inverse: one step of iterative
// refinement of batched inverses,
//   X <- X + X (I - A X),
// with the residual I - A X accumulated in FP64 (products of two FP32 values
// are exact in FP64, so only the n-term sums round) and the correction
// X (I - A X) formed by FP32 MFMA and added to X with one rounding, alone or
// fused into the inversion (lu_refined.hpp).  The reference has no
// refinement: its inverse is the FP32 LU result itself (parallel_pivot/
// luBatchedInplace.cuh:84-125), and its check only counts matrices within
// 1e-3 of I (verify.hpp:50-103).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "lub_internal.h"
#include "lubatch.h"

namespace {

int check_args(const float* A, float* X, int n, int64_t batch) {
  if (n < 1 || n > LUB_MAX_N) return LUB_EINVAL_N;
  if (batch < 0) return LUB_EINVAL_BATCH;
  if (batch == 0) return LUB_OK;
  if (A == nullptr || X == nullptr) return LUB_ENULL;
  if ((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(X)) & 3) return LUB_EALIGN;
  return -1;  // proceed
}

// One workgroup per tile (several tiles per workgroup measured slower).
int enqueue(const void* fn, int layout, const float* A, float* X, int* piv, int64_t batch, void* stream) {
  if (fn == nullptr) return LUB_ENODEVICE;
  const int per_tile = 64 / lub::kLayoutLanes[layout];  // matrices
  int64_t ntiles = (batch + per_tile - 1) / per_tile;
  const unsigned grid = static_cast<unsigned>(std::min<int64_t>(ntiles, int64_t(1) << 22));
  int vec = ((reinterpret_cast<uintptr_t>(A) & 15u) == 0 ? 1 : 0) | ((reinterpret_cast<uintptr_t>(X) & 15u) == 0 ? 2 : 0);
  void* args[] = {&A, &X, &piv, &batch, &ntiles, &vec};
  return hipLaunchKernel(fn, dim3(grid), dim3(64), args, 0, static_cast<hipStream_t>(stream)) == hipSuccess ? LUB_OK
                                                                                                        : LUB_EHIP;
}

}  // namespace

extern "C" {

int lu_batched_refine(const float* A, float* X, int n, int64_t batch, void* stream) {
  const int rc = check_args(A, X, n, batch);
  if (rc >= 0) return rc;
  const bool quads = n <= lub::kRefineQuadMaxN && !lub::rows_beat_quads(n, false, batch, lub::kSmallBatchRefinedQuads);
  const int layout = quads ? 1 : 0;
  return enqueue(lub::kernel_table().refine[n][layout], layout, A, X, nullptr, batch, stream);
}

int lu_batched_inverse_refined(const float* A, float* X, int* piv, int n, int64_t batch, int flags, void* stream) {
  const int rc = check_args(A, X, n, batch);
  if (rc >= 0) return rc;
  if (A == X) return LUB_EINVAL_ARG;  // A must survive for the residual
  const int rule = flags & LUB_PIVOT_MASK, layout = flags & LUB_LAYOUT_MASK;
  if ((flags & ~(LUB_PIVOT_MASK | LUB_LAYOUT_MASK)) != 0 || rule > LUB_PIVOT_GEPP || layout == LUB_LAYOUT_MASK ||
      (layout == LUB_LAYOUT_QUAD4 && n > lub::kLayoutMaxN[1]))
    return LUB_EFLAGS;
  const bool any_piv = n >= 17 && (rule == LUB_PIVOT_NONE || rule == LUB_PIVOT_PARALLEL || rule == LUB_PIVOT_SERIAL);
  if (!any_piv && (reinterpret_cast<uintptr_t>(piv) & 3u) != 0) return LUB_EALIGN;
  const int chosen = lub::choose_layout(n, flags, batch, lub::kSmallBatchRefinedQuads);
  return enqueue(lub::kernel_table().refined[n][rule][chosen], chosen, A, X, piv, batch, stream);
}

}  // extern "C"
