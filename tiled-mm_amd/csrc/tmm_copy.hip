// Copies of many small matrices between page-locked host memory and the device by one kernel (gfx950).
//
// A DMA command costs about 10 us beside its transfer (64 KB at 6 GB/s, 1 MB at 38), and a batch of
// small matrices issues three per problem. A kernel reads and writes page-locked memory over the same
// link at its full rate (64 MB at 56.7 GB/s from 64 workgroups, 55.2 GB/s back from 32; DMA 57.0), so
// that one launch copies the matrices of a group. Bound by the link; a thread keeps 8 accesses in
// flight, 32 KB per workgroup, and 64 workgroups leave the CUs to the tile kernels beside them (256
// and more ran slower: 53 GB/s).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "tmm_kernels.h"

namespace tmm {
namespace {

typedef double d2 __attribute__((ext_vector_type(2)));
constexpr int kThreads = 256, kInFlight = 8;  // accesses of a thread in flight

// count units of src to dst; at(i): position of unit i in each
template <typename V, typename At>
__device__ __forceinline__ void copy_units(const V* __restrict__ src, V* __restrict__ dst, int count, At at) {
  for (int i0 = threadIdx.x; i0 < count; i0 += kThreads * kInFlight) {
    V v[kInFlight];
    long to[kInFlight];
#pragma unroll
    for (int u = 0; u < kInFlight; ++u) {
      const int i = i0 + u * kThreads;
      if (i < count) {
        long from;
        at(i, from, to[u]);
        v[u] = src[from];
      }
    }
#pragma unroll
    for (int u = 0; u < kInFlight; ++u)
      if (i0 + u * kThreads < count) dst[to[u]] = v[u];
  }
}

__global__ __launch_bounds__(kThreads) void copy_items_kernel(const CopyItem* __restrict__ items, int n) {
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "");  // what the host wrote, also to memory that the L2 may hold
  for (int t = blockIdx.x; t < n; t += gridDim.x) {
    const CopyItem it = items[t];
    const int count = it.rows * it.cols;
    if (it.ld_src == it.rows && it.ld_dst == it.rows && !(((uintptr_t)it.src | (uintptr_t)it.dst) & 15)) {
      copy_units((const d2*)it.src, (d2*)it.dst, count / 2, [](int i, long& from, long& to) { from = to = i; });
      if ((count & 1) && threadIdx.x == 0) it.dst[count - 1] = it.src[count - 1];
    } else {
      copy_units(it.src, it.dst, count, [&](int i, long& from, long& to) {
        const int c = i / it.rows, r = i - c * it.rows;
        from = r + c * it.ld_src;
        to = r + c * it.ld_dst;
      });
    }
  }
}

}  // namespace

hipError_t launch_copy_items(const CopyItem* items, int n, int workgroups, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(copy_items_kernel, dim3(n < workgroups ? n : workgroups), dim3(kThreads), 0, s, items, n);
  return hipGetLastError();
}

}  // namespace tmm
