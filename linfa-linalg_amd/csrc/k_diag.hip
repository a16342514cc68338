// Fast factor + inverse of 64 x 64 diagonal blocks (the device code is in
// k_diag_impl.h) for a grouped batch step: one workgroup per (system, block).
#include "k_diag_impl.h"
#include "k_subst_impl.h"
#include "llh_kernels.h"

namespace llh {
namespace {

// Grouped form for the batch planner: work w = (item, k0) factors and inverts
// the block at (k0, k0) of its system; a failure sets the system's status.
// With a forward workspace (bb.y) it also takes the block's forward step.  Three
// workgroups per CU: bounded to four, f64 spills registers (the 20000-system batch
// 8.99 against 8.53 ms).
template <typename T>
__global__ __launch_bounds__(kDiagT, 3) void grp_diag_fast_kernel(const BatchBase<T>* __restrict__ base,
                                                           const BatchItem* __restrict__ items,
                                                           const StepWork* __restrict__ work, int count) {
  if ((int)blockIdx.x >= count) return;
  const StepWork w = work[blockIdx.x];
  const BatchItem it = items[w.item];
  const BatchBase<T> bb = *base;
  int32_t* st = bb.status + it.id;
  __shared__ __attribute__((aligned(16))) DiagLds<T> sm;
  if (threadIdx.x == 0) sm.skip = *st != kNoFail;
  __syncthreads();
  if (sm.skip) return;
  const bool fwd = bb.y != nullptr;
  FwdDiagPrefetch<T> f{};
  if (fwd) f = fwd_diag_prefetch<T>(bb, it, w.k0);
  if (diag_quad_block<T, T>(bb.a + it.a_off + (int64_t)w.k0 * it.lda + w.k0, it.lda, min(kNB, it.n - w.k0),
                            bb.linv + it.linv_off + (int64_t)(w.k0 / kNB) * kNB * kNB, st, w.k0, sm))
    return;
  if (fwd) {
    __syncthreads();  // the inverse is stored; the block's LDS is free
    static_assert(sizeof(sm.l) >= kNB * (kNB + 1) * sizeof(T) && sizeof(sm.x) >= kNB * kSolveCols * sizeof(T),
                  "the forward step's tiles fit the block's LDS");
    grp_forward_diag<T>(bb, it, w.k0, sm.l, sm.x, f);
  }
}

}  // namespace

template <typename T>
hipError_t launch_grp_diag_fast(const BatchBase<T>* base, const BatchItem* items, const StepWork* work,
                                int count, hipStream_t s) {
  if (count <= 0) return hipSuccess;
  hipLaunchKernelGGL((grp_diag_fast_kernel<T>), dim3(count), dim3(kDiagT), 0, s, base, items, work, count);
  return hipGetLastError();
}
template hipError_t launch_grp_diag_fast<double>(const BatchBase<double>*, const BatchItem*, const StepWork*,
                                                 int, hipStream_t);
template hipError_t launch_grp_diag_fast<float>(const BatchBase<float>*, const BatchItem*, const StepWork*, int,
                                                hipStream_t);

}  // namespace llh
