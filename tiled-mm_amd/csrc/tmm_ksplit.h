// Tile kernels with the inner dimension split over a workgroup's waves: launch interface, and the
// choice between their tile shapes and the 128 x 128 (complex double: 64 x 64) pipelined kernels.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <limits>

#include "tmm_kernels.h"

namespace tmm {

// Element types as the tables below order them.
enum class KsType { D = 0, S = 1, Z = 2, C = 3 };

// Tile shapes in blocks of 16 rows and columns, and the ring stages of each. Two stages where that
// lets more workgroups share a CU (a third one ran 2-4% slower at 2048^3); the smallest shapes have
// so little work per stage that they take four. Complex double stops at 3 x 3 and complex float
// at 3 x 4: larger tiles exceed the 256 registers of two waves per SIMD.
#define TMM_KS_SHAPES_SMALL(X, S23) \
  X(1, 1, 4) X(1, 2, 4) X(2, 1, 4) X(2, 2, 2) X(2, 3, S23) X(3, 2, S23) X(3, 3, 2)
#define TMM_KS_SHAPES_MIDDLE(X) X(2, 4, 2) X(4, 2, 2) X(3, 4, 2) X(4, 3, 2)
#define TMM_KS_SHAPES_LARGE(X) X(4, 4, 2)

struct KsShape {
  int m, n;
};
#define TMM_KS_ENTRY(a, b, s) {a, b},
constexpr KsShape kKsShapes[] = {TMM_KS_SHAPES_SMALL(TMM_KS_ENTRY, 3) TMM_KS_SHAPES_MIDDLE(TMM_KS_ENTRY)
                                     TMM_KS_SHAPES_LARGE(TMM_KS_ENTRY)};
#undef TMM_KS_ENTRY
constexpr int kKsShapeCount[4] = {12, 12, 7, 11};  // shapes of each element type, a prefix of kKsShapes

struct KsCost {  // a type's costs; cycles of a 2.4 GHz clock
  int bk;        // inner dimension of a stage
  int block;     // a wave's MFMA cycles per stage and 16 x 16 block
  int stage;     // what a stage costs beside its MFMAs
  int pipe;      // the same of a k-step of the pipelined kernel
  int pipe_bk;   // inner dimension of that k-step (16 blocks per wave; complex double: 8 of half the size)
  double tile;   // us per block of a tile's prologue and epilogue
};
// Fitted to the times of every shape at about 20 sizes from 17 x 33 x 5 to 6222 x 6255 x 3501 (the
// choice they lead to is within 3% of the fastest shape at each of them; over 180 random products, those of
// short_inner aside, 1 to 3% behind it on average and 25% at worst).
constexpr KsCost kKsCost[4] = {{8, 128, 170, 150, 8, 0.28},
                               {16, 128, 280, 290, 16, 0.26},
                               {4, 256, 170, 250, 8, 0.78},
                               {8, 256, 300, 385, 8, 0.33}};

// Time in us of a product of (together) `tiles` tiles of shape s and inner dimension k on `cus`
// compute units: whole tiles per CU, four waves sharing a tile's stages.
inline double ks_time(KsType t, KsShape s, long tiles, long k, int cus) {
  const KsCost& c = kKsCost[(int)t];
  const int blocks = s.m * s.n;
  // a stage cannot run faster than the L2 delivers it (about 24 bytes per cycle and CU), which
  // binds for the smallest tiles; 12 complex float blocks leave fewer registers to overlap with
  const double extra = t == KsType::C && blocks == 12 ? 240 : 0;
  double per = std::max(blocks * c.block + c.stage + extra, (s.m + s.n) * 4096 / 24.0);
  // With many tiles per CU and a long inner dimension the workgroups of an XCD drift apart in k and
  // share less in its L2: at four or more tiles per CU the real types lose up to 8% from 24 KB to
  // 64 KB of inner dimension (FP64 TN 5000^3 3.74 ms against 3.61 without the loss, 6000 x 6000 x
  // 8000 8.73 against 8.09).
  if (t <= KsType::S && tiles > 4L * cus) {
    const double kb = k * (t == KsType::D ? 8.0 : 4.0);
    per *= 1 + 0.08 * std::min(1.0, std::max(0.0, (kb - 24000) / 40000));
  }
  return 2.3 + c.tile * blocks + (double)((tiles + cus - 1) / cus) * ((double)k / c.bk / 4) * per / 2400;
}
// The same for `tiles` workgroup tiles of the pipelined kernel.
inline double pipe_time(KsType t, long tiles, long k, int cus) {
  const KsCost& c = kKsCost[(int)t];
  const int step = t == KsType::Z ? 8 * c.block : 16 * c.block;  // a wave's MFMA cycles per k-step
  return 2.3 + 4 * c.tile + (double)((tiles + cus - 1) / cus) * ((double)k / c.pipe_bk) * (step + c.pipe) / 2400;
}

inline long ks_tiles(KsShape s, long m, long n) { return ((m + 16 * s.m - 1) / (16 * s.m)) * ((n + 16 * s.n - 1) / (16 * s.n)); }

// Tiles of one launch: a grid holds fewer than 2^32 threads, 256 per tile. The largest C's that fit the device have more
// small tiles than that (131072 x 131072, 69 GB in FP32, has 2^24 of 32 x 32; so has a C of 2^29 x 1 in 32 x 16).
constexpr long kKsMaxTiles = (1L << 24) - 1;

// Fastest shape for an m x n x k product, and its time in us (infinite if none has few enough tiles).
inline int ks_shape(KsType t, long m, long n, long k, int cus, double* us) {
  int best = 0;
  double least = std::numeric_limits<double>::infinity();
  for (int i = 0; i < kKsShapeCount[(int)t]; ++i) {
    const long tiles = ks_tiles(kKsShapes[i], m, n);
    if (tiles > kKsMaxTiles) continue;
    const double x = ks_time(t, kKsShapes[i], tiles, k, cus);
    if (x < least) {
      least = x;
      best = i;
    }
  }
  *us = least;
  return best;
}

// Time in us of a product on the faster of the two kernels.
inline double product_time(KsType t, long m, long n, long k, int cus) {
  double us = 0;
  ks_shape(t, m, n, k, cus, &us);
  const long edge = t == KsType::Z ? 64 : 128, tiles = ((m + edge - 1) / edge) * ((n + edge - 1) / edge);
  return tiles >= 2L * cus ? std::min(us, pipe_time(t, tiles, k, cus)) : us;
}

// Products with a short inner dimension and more than two 32 x 32 tiles per CU (no side within one of 16): the times above count a tile's
// first loads and its C once per product, which is right for a long inner dimension or few tiles; here they
// are most of the work of every tile. Kernel by kernel, in us: a product, every round of its tiles over
// the CUs, and each k of a round. Fitted to 50 products per type without and 50 with a C that is read, from 399 x 4207 to
// 6874 x 1710 with k from 1 on (4 to 16% rms); the choice they lead to is 0.5 to 2.5% behind the fastest kernel on
// average (complex double with a C read 4%). With the times above 16 x 16 tiles were taken for the shortest: in us, with
// these / with those, SGEMM 2000 x 2000 x 1 9.8 / 27, 6000 x 6000 x 1 36 / 160; DGEMM 2000 x 2000 x 1 12.3 / 28, x 64
// 19.6 / 24.4, 6000 x 6000 x 8 67 / 89; ZGEMM 6000 x 6000 x 64 308 / 419; CGEMM 2000 x 2000 x 64 25 / 31; near the upper
// end SGEMM 3073 x 6846 x 309 139 / 169, DGEMM 4258 x 1250 x 144 41 / 50, ZGEMM 3941 x 5734 x 187 531 / 587.
struct ShortCost {
  double product, round, k;
};
enum class ShortKernel { Ks32, Pipe, Real };  // 32 x 32 k-split, pipelined, register-staged tiles
constexpr int kShortMaxK[4] = {160, 512, 256, 128};  // above, the times further up choose as well or better
constexpr int kShortShape = 3;  // 32 x 32 in kKsShapes
inline bool short_inner(KsType t, long m, long n, long k, int cus) {
  const long tiles = ks_tiles(kKsShapes[kShortShape], m, n);
  return k <= kShortMaxK[(int)t] && m > 16 && n > 16 && tiles > 2L * cus && tiles <= kKsMaxTiles;
}
// reads_c: beta or an accumulation reads C, which the large tiles do with too little in flight: only complex double's
// (64 x 64) can win then.
inline ShortKernel short_kernel(KsType t, long m, long n, long k, bool reads_c, int cus) {
  constexpr ShortCost ks[4] = {{3.9, 0.70, 0.0068}, {3.8, 0.63, 0.0036}, {4.0, 1.06, 0.0266}, {3.6, 0.79, 0.0136}};
  constexpr ShortCost pipe[4] = {{8.9, 8.3, 0.118}, {5.5, 3.4, 0.057}, {3.2, 2.6, 0.106}, {4.6, 6.1, 0.220}};
  constexpr ShortCost real_d = {4.3, 6.6, 0.128};  // stores its C faster than the pipelined kernel
  constexpr ShortCost ks_zc = {3.3, 1.67, 0.026}, pipe_zc = {5.5, 5.8, 0.1035};
  if (reads_c && t != KsType::Z) return ShortKernel::Ks32;
  auto time = [&](const ShortCost& c, long edge) {
    const long rounds = (((m + edge - 1) / edge) * ((n + edge - 1) / edge) + cus - 1) / cus;
    return c.product + rounds * (c.round + k * c.k);
  };
  const double a = time(reads_c ? ks_zc : ks[(int)t], 32);
  const double b = time(reads_c ? pipe_zc : pipe[(int)t], t == KsType::Z ? 64 : 128);
  if (t == KsType::D && time(real_d, 128) < std::min(a, b)) return ShortKernel::Real;
  return b < a ? ShortKernel::Pipe : ShortKernel::Ks32;
}

// Whether an operand's 16-byte row chunks reach over the end of at most one column (a chunk of 4
// floats over the end of a column, or of two complex floats, of a leading dimension below its size).
template <typename R>
bool ks_chunks_ok(bool cplx, bool kc, long rows, long ld) {
  const long chunk = 16 / ((long)sizeof(R) * (cplx ? 2 : 1));
  return kc || rows % chunk == 0 || ld >= chunk - 1;
}
// Whether the kernels take the product: a lane's byte offsets inside a load (up to 15 rows or
// columns) are 32 bits wide.
template <typename R>
bool ks_takes(const GemmParams<R>& p, bool cplx) {
  const long es = (long)sizeof(R) * (cplx ? 2 : 1);
  return p.variant == 1 && p.k > 0 && p.lda * es <= (1L << 28) && p.ldb * es <= (1L << 28) &&
         ks_chunks_ok<R>(cplx, p.opa != 'N', p.m, p.lda) && ks_chunks_ok<R>(cplx, p.opb == 'N', p.n, p.ldb);
}

// A product whose tiles are shared by several workgroups ("parts"), for a C of fewer tiles than the
// CUs take and a long inner dimension: without the split most CUs idle (500 x 600 in 32 x 48 tiles: 208
// for 256 CUs, and a fifth of each stage beside its MFMAs) or a few run alone. Each part's m x n sums
// go through device memory, and a second kernel adds them: about 5.5 us for the two launches and the
// events that order the buffer, and 2.5 MB of sums per us. (Adding them up in the last workgroup of a
// tile to arrive, in one launch, took 20 to 150 us more: one workgroup reads a tile's sums.)
// Unsplit -> split in us: DGEMM TN 500 x 600 x 40000 478 -> 397, NN 32 x 32 x 20000 64 -> 10, TN 100 x
// 100 x 10000 33 -> 14, NT 300 x 700 x 15000 135 -> 111; SGEMM TN 500 x 600 x 40000 247 -> 212; ZGEMM NN
// 500 x 300 x 10000 312 -> 237 (210 in 32 x 32 tiles), CN 200 x 200 x 5000 55 -> 41.
constexpr int kSplitShapes[4] = {0, 3, 6, 11};  // 16 x 16, 32 x 32, 48 x 48, 64 x 64 (the real types)
constexpr long kSplitMaxWorkgroups = 512;
// Bytes that the sums of every split product of the type fit in.
inline size_t split_bytes(KsType t) {
  const size_t es[4] = {8, 4, 16, 8};
  const size_t edge = t <= KsType::S ? 64 : 48;
  return kSplitMaxWorkgroups * edge * edge * es[(int)t];
}
struct SplitPlan {
  int shape, parts;  // parts < 2: not split
};
// The fastest split of an m x n x k product where the model gives it a lead of 4.5 us (it is that far
// out for an unsplit product of a few small tiles: SGEMM TN 64 x 64 x 4000 runs in 8.4 us unsplit, not
// 13.2, and 9.6 split); one or two workgroups per CU (one leaves its waits uncovered: 3%), and 8 stages
// at least for every wave.
inline SplitPlan split_plan(KsType t, long m, long n, long k, int cus) {
  SplitPlan best = {0, 1};
  const KsCost& c = kKsCost[(int)t];
  const double es[4] = {8, 4, 16, 8};
  if (k < 64 * c.bk) return best;
  double least = product_time(t, m, n, k, cus) - 4.5;
  for (int shape : kSplitShapes) {
    if (shape >= kKsShapeCount[(int)t]) continue;
    const KsShape s = kKsShapes[shape];
    const long tiles = ks_tiles(s, m, n);
    for (long slots : {2L * cus, (long)cus}) {
      const long parts = std::min({slots / tiles, kSplitMaxWorkgroups / tiles, k / (32 * c.bk)});
      if (parts < 2) continue;
      const double us = ks_time(t, s, tiles * parts, (k + parts - 1) / parts, cus) * (tiles * parts <= cus ? 1.03 : 1) +
                        5.5 + parts * m * n * es[(int)t] / 2.5e6;
      if (us < least) {
        least = us;
        best = {shape, (int)parts};
      }
    }
  }
  return best;
}

// One product on the given shape (an index of kKsShapes), or a group of products with one op pair,
// alpha and k in one launch; every product must satisfy ks_takes. The result does not depend on
// the shape, nor on the grouping.
#define TMM_KS_DECLARE(t, R)                                                   \
  hipError_t launch_ks_##t(const GemmParams<R>& p, int shape, hipStream_t s); \
  hipError_t launch_ks_##t##_group(const GemmParams<R>* tiles, int count, hipStream_t s); \
  hipError_t launch_ks_##t##_split(const GemmParams<R>& p, int shape, int parts, void* ws, hipStream_t s);
TMM_KS_DECLARE(d, double)
TMM_KS_DECLARE(s, float)
TMM_KS_DECLARE(z, double)
TMM_KS_DECLARE(c, float)
#undef TMM_KS_DECLARE
// A batch of products as launch_gemm_d_batched describes it, in 64 x 64 tiles.
hipError_t launch_ks_d_batched(char opa, char opb, const GemmParams<double>* probs, const int* items, int n_items,
                               int* counter, int n_workgroups, hipStream_t s);

}  // namespace tmm
