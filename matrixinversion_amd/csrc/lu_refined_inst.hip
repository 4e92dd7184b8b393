// lu_refined_inst.hip -- instantiates lu_refined_kernel<N, L, PIV> (inverse +
// one refinement step in one kernel, and the refinement of a given inverse)
// for N in [LUB_RF_LO, LUB_RF_HI], every pivot rule and the layouts of the
// plain kernel (16-lane rows, quads up to n = 16), and registers the host
// handles.  Compiled once per size range so the units build in parallel.
#include "lu_refined.hpp"
#include "lub_internal.h"

#ifndef LUB_RF_LO
#error "LUB_RF_LO / LUB_RF_HI must be defined"
#endif

#define LUB_RCAT3(a, b, c) a##b##_##c
#define LUB_RCATX(a, b, c) LUB_RCAT3(a, b, c)
#define LUB_RF_REGISTER_NAME LUB_RCATX(lub_register_refined_, LUB_RF_LO, LUB_RF_HI)

namespace {

template <int N, int L, int PIV>
const void* handle() {
  return reinterpret_cast<const void*>(&lub::lu_refined_kernel<N, L, PIV>);
}

template <int N, int L>
void register_layout(lub::KernelTable* t, int layout) {
  auto& slot = t->refined[N];
  slot[lub::kPivNone][layout] = handle<N, L, lub::kPivNone>();
  slot[lub::kPivParallel][layout] = handle<N, L, lub::kPivParallel>();
  slot[lub::kPivSerial][layout] = slot[lub::kPivParallel][layout];  // the same pivots
  slot[lub::kPivTree][layout] = handle<N, L, lub::kPivTree>();
  slot[lub::kPivGepp][layout] = handle<N, L, lub::kPivGepp>();
}

template <int N>
void register_range(lub::KernelTable* t) {
  if constexpr (N <= LUB_RF_HI) {
    register_layout<N, 16>(t, 0);
    if constexpr (N <= lub::kLayoutMaxN[1]) register_layout<N, 4>(t, 1);
    // the two that lu_batched_refine picks from
    if constexpr (N > lub::kGeppQuadMaxN) t->refine[N][0] = handle<N, 16, lub::kPivGiven>();
    if constexpr (N <= lub::kRefineQuadMaxN) t->refine[N][1] = handle<N, 4, lub::kPivGiven>();
    register_range<N + 1>(t);
  }
}

}  // namespace

extern "C" void LUB_RF_REGISTER_NAME(lub::KernelTable* t) { register_range<LUB_RF_LO>(t); }
