// Complex double instances of the kernels that split the inner dimension over a workgroup's waves.
#include "tmm_ksplit_kernel.h"

namespace tmm {

hipError_t launch_ks_z(const GemmParams<double>& p, int shape, hipStream_t s) {
  int i = 0;
#define TMM_KS_CASE(a, b, st) \
  if (shape == i++) return ks::launch_shape<ks::TypeZ, a, b, st>(p, s);
  TMM_KS_SHAPES_SMALL(TMM_KS_CASE, 2)
#undef TMM_KS_CASE
  return hipErrorInvalidValue;
}

hipError_t launch_ks_z_group(const GemmParams<double>* tiles, int count, hipStream_t s) {
  return ks::launch_group<ks::TypeZ, 3, 3, 2>(tiles, count, s);
}

hipError_t launch_ks_z_split(const GemmParams<double>& p, int shape, int parts, void* ws, hipStream_t s) {
  if (shape == kSplitShapes[0]) return ks::launch_split<ks::TypeZ, 1, 1, 4>(p, parts, ws, s);
  if (shape == kSplitShapes[1]) return ks::launch_split<ks::TypeZ, 2, 2, 2>(p, parts, ws, s);
  if (shape == kSplitShapes[2]) return ks::launch_split<ks::TypeZ, 3, 3, 2>(p, parts, ws, s);
  return hipErrorInvalidValue;
}

}  // namespace tmm
