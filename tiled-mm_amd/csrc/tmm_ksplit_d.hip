// Double instances of the kernels that split the inner dimension over a workgroup's waves.
#include "tmm_ksplit_kernel.h"

namespace tmm {

hipError_t launch_ks_d(const GemmParams<double>& p, int shape, hipStream_t s) {
  int i = 0;
#define TMM_KS_CASE(a, b, st) \
  if (shape == i++) return ks::launch_shape<ks::TypeD, a, b, st>(p, s);
  TMM_KS_SHAPES_SMALL(TMM_KS_CASE, 3)
  TMM_KS_SHAPES_MIDDLE(TMM_KS_CASE)
  TMM_KS_SHAPES_LARGE(TMM_KS_CASE)
#undef TMM_KS_CASE
  return hipErrorInvalidValue;
}

hipError_t launch_ks_d_group(const GemmParams<double>* tiles, int count, hipStream_t s) {
  return ks::launch_group<ks::TypeD, 4, 4, 2>(tiles, count, s);
}

hipError_t launch_ks_d_batched(char opa, char opb, const GemmParams<double>* probs, const int* items, int n_items,
                               int* counter, int n_workgroups, hipStream_t s) {
  const dim3 grid(std::min(n_items, n_workgroups)), block(256);
  const bool akc = opa != 'N', bkc = opb == 'N';
  if (akc && bkc) hipLaunchKernelGGL((ks::gemm_ks_batched_kernel<ks::TypeD, true, true, 4, 4, 2>), grid, block, 0, s, probs, items, n_items, counter);
  else if (akc) hipLaunchKernelGGL((ks::gemm_ks_batched_kernel<ks::TypeD, true, false, 4, 4, 2>), grid, block, 0, s, probs, items, n_items, counter);
  else if (bkc) hipLaunchKernelGGL((ks::gemm_ks_batched_kernel<ks::TypeD, false, true, 4, 4, 2>), grid, block, 0, s, probs, items, n_items, counter);
  else hipLaunchKernelGGL((ks::gemm_ks_batched_kernel<ks::TypeD, false, false, 4, 4, 2>), grid, block, 0, s, probs, items, n_items, counter);
  return hipGetLastError();
}

hipError_t launch_ks_d_split(const GemmParams<double>& p, int shape, int parts, void* ws, hipStream_t s) {
  if (shape == kSplitShapes[0]) return ks::launch_split<ks::TypeD, 1, 1, 4>(p, parts, ws, s);
  if (shape == kSplitShapes[1]) return ks::launch_split<ks::TypeD, 2, 2, 2>(p, parts, ws, s);
  if (shape == kSplitShapes[2]) return ks::launch_split<ks::TypeD, 3, 3, 2>(p, parts, ws, s);
  if (shape == kSplitShapes[3]) return ks::launch_split<ks::TypeD, 4, 4, 2>(p, parts, ws, s);
  return hipErrorInvalidValue;
}

}  // namespace tmm
