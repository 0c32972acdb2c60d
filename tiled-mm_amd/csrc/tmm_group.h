// Grouped launches: the descriptor's host side and the device side's look-up.
#pragma once
#include <hip/hip_runtime.h>

#include "tmm_kernels.h"

namespace tmm {

// The product of a grouped launch that workgroup w works on, with its parameters; -1 for a padding
// workgroup. Products start on multiples of 8 workgroups, so that a workgroup's XCD
// (blockIdx.x % 8) is the one its tile order assumes.
template <typename R>
__device__ __forceinline__ int group_member(const TileGroup<R>& g, int w, int tiles_m, int tiles_n,
                                            GemmParams<R>& prm, int& local) {
  int t = 0;
  while (t + 1 < g.count && w >= g.wg_start[t + 1]) ++t;
  prm = g.base;
  prm.m = g.m[t];
  prm.n = g.n[t];
  prm.a = g.a[t];
  prm.lda = g.lda[t];
  prm.b = g.b[t];
  prm.ldb = g.ldb[t];
  prm.c = g.c[t];
  prm.ldc = g.ldc[t];
  prm.cin = g.cin[t];
  prm.ldcin = g.ldcin[t];
  prm.beta = g.beta[t];
  prm.beta_im = g.beta_im[t];
  prm.accumulate = g.accumulate[t];
  local = w - g.wg_start[t];
  const int nbm = (prm.m + tiles_m - 1) / tiles_m, nbn = (prm.n + tiles_n - 1) / tiles_n;
  return local < nbm * nbn ? t : -1;
}

// The descriptor of `count` products with one op pair, alpha and k; false if they do not form a
// group. edge_m, edge_n: rows and columns of C per workgroup of the group's kernel.
template <typename R>
bool make_group(const GemmParams<R>* tiles, int count, int edge_m, int edge_n, TileGroup<R>& g, int& wg) {
  if (count <= 0 || count > kDgemmGroupMax) return false;
  g = TileGroup<R>{};
  g.base = tiles[0];
  g.count = count;
  wg = 0;
  for (int t = 0; t < count; ++t) {
    const GemmParams<R>& p = tiles[t];
    if (p.k != g.base.k || p.opa != g.base.opa || p.opb != g.base.opb || p.alpha != g.base.alpha ||
        p.alpha_im != g.base.alpha_im)
      return false;
    g.wg_start[t] = wg;
    wg += (((p.m + edge_m - 1) / edge_m) * ((p.n + edge_n - 1) / edge_n) + 7) / 8 * 8;
    g.m[t] = p.m;
    g.n[t] = p.n;
    g.a[t] = p.a;
    g.lda[t] = p.lda;
    g.b[t] = p.b;
    g.ldb[t] = p.ldb;
    g.c[t] = p.c;
    g.ldc[t] = p.ldc;
    g.cin[t] = p.cin;
    g.ldcin[t] = p.ldcin;
    g.beta[t] = p.beta;
    g.beta_im[t] = p.beta_im;
    g.accumulate[t] = p.accumulate;
  }
  g.wg_start[count] = wg;
  return true;
}

}  // namespace tmm
