// Tile kernels that split the inner dimension over the waves of a workgroup (gfx950).
//
// For products whose 128 x 128 workgroup tiles do not fill the device. A workgroup owns a small
// C tile (16 to 64 rows and columns) and each of its four waves computes the whole tile over a
// quarter of the inner dimension (k-steps dealt out in turn), so that even a small C keeps every
// SIMD of its CU busy and a long inner dimension is four times shorter per wave. A wave fills and
// reads an LDS ring of its own with direct global->LDS loads: the main loop has no barrier. The
// four partial tiles meet in LDS, in a fixed order, in front of the fused epilogue.
//
// One template serves the four element types. A stage holds 64 bytes of inner dimension of every
// operand row (8 double, 16 float, 4 complex double, 8 complex float), and a lane's 16-byte
// fragment KV = 2, 4, 1, 2 consecutive values of its row:
//   k-contiguous operand (A for 'T' / 'C', B for 'N'): LDS [row][slot], a wave load fills 16 rows
//     of 64 bytes, chunk q of row r in slot q ^ ((r >> 1) & 3) (conflict-free fragment reads);
//   row-contiguous operand: LDS [k][row], a 16-byte chunk = KV consecutive rows at one k.
// Any m, n, k >= 1: rows beyond the matrix read a clamped in-bounds row (they feed only unstored
// outputs); the last k-step, where it is partial or where a row-contiguous chunk could reach past
// the end of the operand, is read first, element by element, straight into fragments.
//
// What bounds them: the matrix cores once every CU has a tile (the rest of a stage, about 170
// cycles FP64 and 280 FP32 beside 2048 of MFMA for 64 x 64 tiles, is the issue of its loads and LDS
// reads and the waits), the L2 -> LDS path for tiles of 16 x 32 and below, and 3-6 us of launch,
// first loads and epilogue for the smallest products. Measured (HIP events, calls back to back)
// against 128 x 128 tiles that each run the whole inner dimension: DGEMM TN 300 x 200 x 260 62 -> 6
// us, NN 1000^3 148 -> 36, NT 1234 x 4567 x 1357 388 -> 238 (64.3 TFLOP/s), TN 500 x 600 x 40000
// 5358 -> 474, TN 2048^3 285 -> 246 (69.9 TFLOP/s), TN 3000^3 1048 -> 787; SGEMM NN 2048^3 500 -> 135
// (126.8 TFLOP/s); CGEMM CN 1500 x 1300 x 2000 516 -> 252; ZGEMM CN 1000 x 1100 x 1200 304 -> 163.
// The error against an 80-bit product halves (1000^3: 1.07e-15 -> 5.5e-16), the sums being four
// times shorter.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "tmm_group.h"
#include "tmm_kernels.h"
#include "tmm_ksplit.h"

namespace tmm {
namespace ks {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef double d2 __attribute__((ext_vector_type(2)));

struct TypeD {
  typedef double R;
  typedef d2 Chunk;
  typedef d4 Acc;
  static constexpr bool CPLX = false;
};
struct TypeS {
  typedef float R;
  typedef f4 Chunk;
  typedef f4 Acc;
  static constexpr bool CPLX = false;
};
struct TypeZ {
  typedef double R;
  typedef d2 Chunk;
  typedef d4 Acc;
  static constexpr bool CPLX = true;
};
struct TypeC {
  typedef float R;
  typedef f4 Chunk;
  typedef f4 Acc;
  static constexpr bool CPLX = true;
};

__device__ __forceinline__ d4 mfma(double a, double b, d4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f4 mfma(float a, float b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
// column within a 16 x 16 block of accumulator register r (operands swapped: instruction rows are
// C columns; the f64 and f32 forms number them differently)
__device__ __forceinline__ int out_col(double, int lane, int r) { return (lane >> 4) + 4 * r; }
__device__ __forceinline__ int out_col(float, int lane, int r) { return 4 * (lane >> 4) + r; }

template <int VM>
__device__ __forceinline__ void wait_vm() {  // at most VM vector loads outstanding
  static_assert(VM >= 0 && VM < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((VM & 15) | ((VM >> 4) << 14) | (7 << 4) | (15 << 8));
}
__device__ __forceinline__ void wait_lds() { __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4)); }

// One operand of a wave's tile: 16 * WB rows of 64 bytes of inner dimension per stage.
template <typename T, bool KC, int WB>
struct Operand {
  typedef typename T::R R;
  typedef typename T::Chunk Chunk;
  static constexpr int ES = (int)sizeof(R) * (T::CPLX ? 2 : 1);  // bytes per element
  static constexpr int KV = 16 / ES;                             // elements per chunk
  static constexpr int BK = 64 / ES;                             // inner dimension of a stage
  static constexpr int ROWS = 16 * WB;
  static constexpr int READS = KC || KV == 1 ? 1 : KV;  // LDS reads of a fragment

  const char* base;   // stage to load next, wave-uniform
  long off[WB];       // bytes from base to each load's first row (or k), wave-uniform
  unsigned voff[WB];  // this lane's bytes from there
  long step;          // bytes between the wave's stages

  __device__ __forceinline__ static int swz(int r) { return (r >> 1) & 3; }

  __device__ __forceinline__ void setup(const R* p, long ld, int r0, int rows, int stage, int stride, int lane) {
    const char* q0 = (const char*)p;
    if (KC) {
      base = q0 + ((long)r0 * ld + (long)stage * BK) * ES;
      step = (long)stride * BK * ES;
#pragma unroll
      for (int t = 0; t < WB; ++t) {
        const int first = min(r0 + t * 16, rows - 1), local = lane >> 2;
        off[t] = (long)(first - r0) * ld * ES;
        voff[t] = (unsigned)(min(r0 + t * 16 + local, rows - 1) - first) * (unsigned)(ld * ES) +
                  16u * ((lane & 3) ^ swz(local));
      }
    } else {
      base = q0 + ((long)r0 + (long)stage * BK * ld) * ES;
      step = (long)stride * BK * ld * ES;
      constexpr int PER_K = ROWS / KV;  // chunks of one k
#pragma unroll
      for (int t = 0; t < WB; ++t) {
        const int c = t * 64 + lane, first = t * 64 / PER_K, kk = c / PER_K - first, row = (c % PER_K) * KV;
        off[t] = (long)first * ld * ES;
        voff[t] = (unsigned)(min(r0 + row, (rows - 1) / KV * KV) - r0) * (unsigned)ES + (unsigned)kk * (unsigned)(ld * ES);
      }
    }
  }
  __device__ __forceinline__ void issue(char* stage) {
#pragma unroll
    for (int t = 0; t < WB; ++t)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(base + off[t] + voff[t]),
                                       (__attribute__((address_space(3))) void*)(stage + t * 1024), 16, 0, 0);
    base += step;
  }
  // fragment of block b: elements k = KV*g .. KV*g + KV-1 of row 16*b + li
  __device__ __forceinline__ static Chunk frag(const char* stage, int b, int li, int lg) {
    if (KC) return *(const Chunk*)(stage + b * 1024 + li * 64 + ((lg ^ swz(li)) << 4));
    Chunk c;
    constexpr int W = 16 / (int)sizeof(R) / KV;  // reals per element
#pragma unroll
    for (int e = 0; e < KV; ++e) {
      const R* q = (const R*)(stage + ((KV * lg + e) * ROWS + b * 16 + li) * ES);
#pragma unroll
      for (int w = 0; w < W; ++w) c[e * W + w] = q[w];
    }
    return c;
  }
  // the same fragment read from global memory, zero from k_end on
  __device__ __forceinline__ static Chunk frag_global(const R* p, long ld, int r0, int rows, int k0, int k_end, int b,
                                                      int li, int lg) {
    Chunk c;
    constexpr int W = 16 / (int)sizeof(R) / KV;
    const int row = min(r0 + b * 16 + li, rows - 1);
#pragma unroll
    for (int e = 0; e < KV; ++e) {
      const int k = k0 + KV * lg + e;
      const R* q = p + (KC ? (long)k + (long)row * ld : (long)row + (long)k * ld) * W;
#pragma unroll
      for (int w = 0; w < W; ++w) c[e * W + w] = k < k_end ? q[w] : R(0);
    }
    return c;
  }
};

template <typename T, int WBM, int WBN>
struct Tile {
  typedef typename T::R R;
  typedef typename T::Chunk Chunk;
  typedef typename T::Acc Acc;
  static constexpr int NACC = T::CPLX ? 2 : 1;
  // MFMAs of half a stage
  static constexpr int HALF = T::CPLX ? WBM * WBN * 16 / (int)sizeof(R) : WBM * WBN * 8 / (int)sizeof(R);
  Acc acc[NACC][WBM][WBN];

  struct Frags {
    Chunk a[WBM], b[WBN];
  };

  __device__ __forceinline__ void zero() {
#pragma unroll
    for (int c = 0; c < NACC; ++c)
#pragma unroll
      for (int i = 0; i < WBM; ++i)
#pragma unroll
        for (int j = 0; j < WBN; ++j) acc[c][i][j] = Acc{0, 0, 0, 0};
  }
  // half 0 and half 1 of a stage's MFMAs. Real: the first and the last of the chunk's k values;
  // complex: the real and the imaginary parts.
  template <int HALF>
  __device__ __forceinline__ void mma(const Frags& f) {
    if constexpr (!T::CPLX) {
      constexpr int KV = 16 / (int)sizeof(R);
#pragma unroll
      for (int e = HALF * KV / 2; e < (HALF + 1) * KV / 2; ++e)
#pragma unroll
        for (int i = 0; i < WBM; ++i)
#pragma unroll
          for (int j = 0; j < WBN; ++j) acc[0][i][j] = mfma(f.b[j][e], f.a[i][e], acc[0][i][j]);
    } else {
      constexpr int KV = 8 / (int)sizeof(R);
#pragma unroll
      for (int e = 0; e < KV; ++e)
#pragma unroll
        for (int i = 0; i < WBM; ++i) {
          const R ar = f.a[i][2 * e], ai = f.a[i][2 * e + 1];
#pragma unroll
          for (int j = 0; j < WBN; ++j) {
            const R br = f.b[j][2 * e], bi = f.b[j][2 * e + 1];
            if constexpr (HALF == 0) {
              acc[0][i][j] = mfma(br, ar, acc[0][i][j]);
              acc[0][i][j] = mfma(bi, -ai, acc[0][i][j]);
            } else {
              acc[1][i][j] = mfma(bi, ar, acc[1][i][j]);
              acc[1][i][j] = mfma(br, ai, acc[1][i][j]);
            }
          }
        }
    }
  }
};

// Instruction order of a stage half: N instructions of class MASK spread evenly over MFMAS MFMAs.
template <int MASK, int N, int MFMAS>
__device__ __forceinline__ void interleave() {
  constexpr int GROUPS = N < MFMAS ? N : MFMAS < 1 ? 1 : MFMAS;
  constexpr int EACH = MFMAS / GROUPS < 1 ? 1 : MFMAS / GROUPS;
#pragma unroll
  for (int g = 0; g < GROUPS; ++g) {
    __builtin_amdgcn_sched_group_barrier(MASK, (N + GROUPS - 1) / GROUPS, 0);
    __builtin_amdgcn_sched_group_barrier(0x008, EACH, 0);
  }
}

template <typename T, int WBM, int WBN, int S>
struct Geometry {
  static constexpr int ES = (int)sizeof(typename T::R) * (T::CPLX ? 2 : 1);
  static constexpr int STAGE = (WBM + WBN) * 1024;  // bytes of a wave's stage
  static constexpr int RING = 4 * S * STAGE;
  static constexpr int COLS16 = 4 * 16 * WBM * 16 * ES;  // the four partial tiles of 16 columns
  static constexpr int JP = RING / COLS16 < 1 ? 1 : RING / COLS16 > WBN ? WBN : RING / COLS16;
  static constexpr int LDS = RING > JP * COLS16 ? RING : JP * COLS16;
};

// A workgroup's share of the inner dimension of a product that is split over workgroups as well.
template <typename R>
struct Part {
  int index, count;
  R* sums;  // this share's m x n sums, without alpha, beta and C
};

// The C tile at (m0, n0). conj_a / conj_b: negate the imaginary part (op 'C'). SPLIT: the
// tile's sums over share part.index of the inner dimension, to part.sums.
template <typename T, bool A_KC, bool B_KC, int WBM, int WBN, int S, bool SPLIT = false>
__device__ __forceinline__ void tile_at(const GemmParams<typename T::R>& prm, bool conj_a, bool conj_b, int m0, int n0,
                                        const Part<typename T::R>& part = {}) {
  typedef typename T::R R;
  typedef Geometry<T, WBM, WBN, S> G;
  typedef Operand<T, A_KC, WBM> OpA;
  typedef Operand<T, B_KC, WBN> OpB;
  typedef Tile<T, WBM, WBN> TileT;
  constexpr int BK = OpA::BK, BM = 16 * WBM, BN = 16 * WBN, PER = WBM + WBN;
  __shared__ __attribute__((aligned(16))) char lds[G::LDS];
  const int M = prm.m, N = prm.n, K = prm.k;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int li = lane & 15, lg = lane >> 4;

  TileT t;
  t.zero();
  // stages read through the ring, and the k range of the step read element by element
  const bool ragged = K % BK != 0 || (!A_KC && M % OpA::KV != 0) || (!B_KC && N % OpB::KV != 0);
  const int nall = ragged ? (K - 1) / BK : K / BK;
  const int first = SPLIT ? (int)((long)nall * part.index / part.count) : 0;
  const int nfull = SPLIT ? (int)((long)nall * (part.index + 1) / part.count) - first : nall;
  const int ns = nfull > wave ? (nfull - wave + 3) / 4 : 0;

  auto conj = [&](typename TileT::Frags& f) {
    if constexpr (T::CPLX) {
      constexpr int KV = 8 / (int)sizeof(R);
      const R sa = conj_a ? R(-1) : R(1), sb = conj_b ? R(-1) : R(1);
#pragma unroll
      for (int e = 0; e < KV; ++e) {
#pragma unroll
        for (int i = 0; i < WBM; ++i) f.a[i][2 * e + 1] *= sa;
#pragma unroll
        for (int j = 0; j < WBN; ++j) f.b[j][2 * e + 1] *= sb;
      }
    }
  };

  OpA oa;
  OpB ob;
  oa.setup(prm.a, prm.lda, m0, M, first + wave, 4, lane);
  ob.setup(prm.b, prm.ldb, n0, N, first + wave, 4, lane);
  char* ring = lds + wave * (S * G::STAGE);
  auto issue = [&](int slot) {
    oa.issue(ring + slot * G::STAGE);
    ob.issue(ring + slot * G::STAGE + WBM * 1024);
  };
  auto read = [&](typename TileT::Frags& f, int slot) {
    const char* st = ring + slot * G::STAGE;
#pragma unroll
    for (int i = 0; i < WBM; ++i) f.a[i] = OpA::frag(st, i, li, lg);
#pragma unroll
    for (int j = 0; j < WBN; ++j) f.b[j] = OpB::frag(st + WBM * 1024, j, li, lg);
  };

  if (ragged && (nfull & 3) == wave && (!SPLIT || part.index == part.count - 1)) {
    typename TileT::Frags f;
#pragma unroll
    for (int i = 0; i < WBM; ++i) f.a[i] = OpA::frag_global(prm.a, prm.lda, m0, M, nall * BK, K, i, li, lg);
#pragma unroll
    for (int j = 0; j < WBN; ++j) f.b[j] = OpB::frag_global(prm.b, prm.ldb, n0, N, nall * BK, K, j, li, lg);
    conj(f);
    t.template mma<0>(f);
    t.template mma<1>(f);
  }
  // A wave without stages (ns = 0) runs through too: it loads nothing, waits for nothing, reads a slot
  // whose contents are not used and multiplies none. With a branch around it the sums after the step
  // above and those after the loop were two sets of registers, and 36 to 516 bytes per lane of
  // the first spilled wherever the tile has 6 complex or 12 blocks and an operand is row-contiguous.
  {
#pragma unroll
    for (int s = 0; s < S; ++s)
      if (s < ns) issue(s);
    if (ns >= S) wait_vm<(S - 1) * PER>();
    else wait_vm<0>();
    typename TileT::Frags f0, f1;
    read(f0, 0);
    int slot = 0;
    // stage i: its fragments are in registers (cur), so its slot takes stage i + S; half of its
    // MFMAs run before the wait for stage i + 1, whose fragments are read under the other half.
    // With one or two waves per SIMD little hides a load's issue time, so the loads go between the
    // MFMAs of the first half and the LDS reads between the first MFMAs of the second.
    auto stage = [&](typename TileT::Frags& cur, typename TileT::Frags& nxt, int i, auto steady) {
      constexpr bool STEADY = decltype(steady)::value;
      const int nslot = slot + 1 == S ? 0 : slot + 1;
      wait_lds();
      __builtin_amdgcn_sched_barrier(0);
      if (STEADY || i + S < ns) issue(slot);
      conj(cur);
      t.template mma<0>(cur);
      if constexpr (STEADY) interleave<0x020, PER, TileT::HALF>();
      __builtin_amdgcn_sched_barrier(0);
      if (STEADY || i + S < ns) wait_vm<(S - 1) * PER>();
      else wait_vm<0>();
      __builtin_amdgcn_sched_barrier(0);
      read(nxt, nslot);  // past the last stage: a slot whose contents are not used
      t.template mma<1>(cur);
      interleave<0x100, WBM * OpA::READS + WBN * OpB::READS, TileT::HALF / 2>();
      __builtin_amdgcn_sched_barrier(0);
      slot = nslot;
    };
    int i = 0;
    for (; i + 1 + S < ns; i += 2) {
      stage(f0, f1, i, std::true_type{});
      stage(f1, f0, i + 1, std::true_type{});
    }
    for (; i + 1 < ns; i += 2) {
      stage(f0, f1, i, std::false_type{});
      stage(f1, f0, i + 1, std::false_type{});
    }
    if (i < ns) stage(f0, f1, i, std::false_type{});
  }

  // The partial tiles, JP column blocks at a time: [wave][column][row] in LDS, then each thread
  // adds the four values of its elements and stores consecutive rows of a column.
  const R alr = prm.alpha, ali = prm.alpha_im, ber = prm.beta, bei = prm.beta_im;
  const bool acc_prev = prm.accumulate != 0, use_cin = ber != R(0) || (T::CPLX && bei != R(0));
  constexpr int NR = T::CPLX ? 2 : 1;
  // U elements per thread and pass, their C loads in flight together: elements x0 + 256 u of the
  // `total` from column n0 + col0 on, their sums from sum(element, component)
  constexpr int U = 4;
  auto store = [&](int x0, int total, int col0, auto sum) {
    long at[U];
    bool ok[U];
    R prev[U][NR], cin[U][NR];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int x = x0 + 256 * u, gi = m0 + x % BM, gj = n0 + col0 + x / BM;
      ok[u] = x < total && gi < M && gj < N;
      at[u] = (long)gi + (long)gj * prm.ldc;
#pragma unroll
      for (int c = 0; c < NR; ++c) prev[u][c] = cin[u][c] = R(0);
    }
    if (acc_prev) {
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int c = 0; c < NR; ++c)
          if (ok[u]) prev[u][c] = prm.c[at[u] * NR + c];
    }
    if (use_cin) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int x = x0 + 256 * u, gi = m0 + x % BM, gj = n0 + col0 + x / BM;
#pragma unroll
        for (int c = 0; c < NR; ++c)
          if (ok[u]) cin[u][c] = prm.cin[((long)gi + (long)gj * prm.ldcin) * NR + c];
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (!ok[u]) continue;
      R* dst = prm.c + at[u] * NR;
      const R xr = sum(u, 0);
      if constexpr (!T::CPLX) {
        R v = alr * xr;
        if (acc_prev) v += prev[u][0];
        if (use_cin) v += ber * cin[u][0];
        dst[0] = v;
      } else {
        const R xi = sum(u, 1);
        R vr = alr * xr - ali * xi, vi = alr * xi + ali * xr;
        if (acc_prev) {
          vr += prev[u][0];
          vi += prev[u][NR - 1];
        }
        if (use_cin) {
          vr += ber * cin[u][0] - bei * cin[u][NR - 1];
          vi += ber * cin[u][NR - 1] + bei * cin[u][0];
        }
        dst[0] = vr;
        dst[1] = vi;
      }
    }
  };
  R* lsum = (R*)lds;
  constexpr int COLS = 16 * G::JP, PART = COLS * BM * NR;  // reals of one wave's part
#pragma unroll
  for (int jp = 0; jp < WBN; jp += G::JP) {
    __syncthreads();  // the ring (first) or the previous columns are no longer read
#pragma unroll
    for (int jj = 0; jj < G::JP; ++jj) {
      if (jp + jj >= WBN) continue;
#pragma unroll
      for (int i = 0; i < WBM; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          R* q = lsum + wave * PART + ((jj * 16 + out_col(R(0), lane, r)) * BM + 16 * i + li) * NR;
          q[0] = t.acc[0][i][jp + jj][r];
          if constexpr (T::CPLX) q[1] = t.acc[1][i][jp + jj][r];
        }
    }
    __syncthreads();
    const int total = min(COLS, BN - 16 * jp) * BM;
    if constexpr (SPLIT) {
      for (int x = threadIdx.x; x < total; x += 256) {
        const int gi = m0 + x % BM, gj = n0 + 16 * jp + x / BM;
        if (gi >= M || gj >= N) continue;
        const R* q = lsum + x * NR;
        R* dst = part.sums + ((long)gi + (long)gj * M) * NR;
#pragma unroll
        for (int c = 0; c < NR; ++c) dst[c] = (q[c] + q[PART + c]) + (q[2 * PART + c] + q[3 * PART + c]);
      }
    } else {
      for (int x0 = threadIdx.x; x0 < total; x0 += 256 * U)
        store(x0, total, 16 * jp, [&](int u, int c) {
          const R* q = lsum + (x0 + 256 * u) * NR + c;
          return (q[0] + q[PART]) + (q[2 * PART] + q[3 * PART]);
        });
    }
  }
}

// Workgroup -> tile: XCD w % 8 takes a contiguous range of tiles, walked in groups of 8 tile rows
// column by column, so that the tiles an XCD runs at one time share operand strips in its L2.
__device__ __forceinline__ void tile_of(int w, int nbm, int nbn, int& bm, int& bn) {
  const int ntiles = nbm * nbn;
  int t = w;
  if (ntiles >= 32) {
    const int xcd = w % 8, per = ntiles / 8, rem = ntiles % 8;
    t = xcd * per + min(xcd, rem) + w / 8;
  }
  const int in_group = 8 * nbn, group = t / in_group, first = group * 8;
  const int gsz = min(nbm - first, 8), r = t - group * in_group;
  bm = first + r % gsz;
  bn = r / gsz;
}

template <typename T, bool A_KC, bool B_KC, int WBM, int WBN, int S>
__device__ __forceinline__ void tile(const GemmParams<typename T::R>& prm, int w) {
  int bm, bn;
  tile_of(w, (prm.m + 16 * WBM - 1) / (16 * WBM), (prm.n + 16 * WBN - 1) / (16 * WBN), bm, bn);
  tile_at<T, A_KC, B_KC, WBM, WBN, S>(prm, prm.opa == 'C', prm.opb == 'C', bm * 16 * WBM, bn * 16 * WBN);
}

template <typename T, bool A_KC, bool B_KC, int WBM, int WBN, int S>
__global__ __launch_bounds__(256, 2) void gemm_ks_kernel(GemmParams<typename T::R> prm) {
  if (prm.gate_a && (*prm.gate_a | *prm.gate_b) == 0) return;  // uniform: before any barrier
  tile<T, A_KC, B_KC, WBM, WBN, S>(prm, blockIdx.x);
}

// Several products in one launch; padding workgroups exit before any barrier.
template <typename T, bool A_KC, bool B_KC, int WBM, int WBN, int S>
__global__ __launch_bounds__(256, 2) void gemm_ks_group_kernel(TileGroup<typename T::R> g) {
  GemmParams<typename T::R> prm;
  int local;
  if (group_member(g, blockIdx.x, 16 * WBM, 16 * WBN, prm, local) < 0) return;
  tile<T, A_KC, B_KC, WBM, WBN, S>(prm, local);
}

// One product whose tiles are each shared by `parts` workgroups; sums: the m x n sums of each share.
// Workgroup w takes, in the XCD order of tile_of, one share of the inner dimension after another: the
// tiles that an XCD runs at one time read the same part of the operands.
template <typename T, bool A_KC, bool B_KC, int WBM, int WBN, int S>
__global__ __launch_bounds__(256, 2) void gemm_ks_split_kernel(GemmParams<typename T::R> prm, int parts,
                                                               typename T::R* __restrict__ sums) {
  constexpr int BM = 16 * WBM, BN = 16 * WBN;
  const int nbm = (prm.m + BM - 1) / BM, tiles = nbm * ((prm.n + BN - 1) / BN), all = tiles * parts;
  const int xcd = blockIdx.x % 8, per = all / 8, rem = all % 8;
  const int i = xcd * per + min(xcd, rem) + blockIdx.x / 8, share = i / tiles, tile = i % tiles;
  const Part<typename T::R> part = {share, parts, sums + (long)share * prm.m * prm.n * (T::CPLX ? 2 : 1)};
  tile_at<T, A_KC, B_KC, WBM, WBN, S, true>(prm, prm.opa == 'C', prm.opb == 'C', tile % nbm * BM, tile / nbm * BN, part);
}

// C from the shares' sums, added in a fixed order: a workgroup takes 64 elements, its four waves a
// quarter of the shares each, 8 loads in flight.
template <typename T>
__global__ __launch_bounds__(256) void split_sum_kernel(GemmParams<typename T::R> prm, int parts,
                                                        const typename T::R* __restrict__ sums) {
  typedef typename T::R R;
  constexpr int NR = T::CPLX ? 2 : 1, U = 8;
  __shared__ R quarter[4][64 * NR];
  const long total = (long)prm.m * prm.n;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const long x = (long)blockIdx.x * 64 + lane;
  const int p0 = (int)((long)parts * wave / 4), p1 = (int)((long)parts * (wave + 1) / 4);
  R acc[NR];
#pragma unroll
  for (int c = 0; c < NR; ++c) acc[c] = R(0);
  if (x < total) {
    for (int p = p0; p < p1; p += U) {
      R v[U][NR];
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int c = 0; c < NR; ++c) v[u][c] = p + u < p1 ? sums[((long)(p + u) * total + x) * NR + c] : R(0);
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int c = 0; c < NR; ++c) acc[c] += v[u][c];
    }
  }
#pragma unroll
  for (int c = 0; c < NR; ++c) quarter[wave][lane * NR + c] = acc[c];
  __syncthreads();
  if (wave != 0 || x >= total) return;
#pragma unroll
  for (int c = 0; c < NR; ++c)
    acc[c] = (quarter[0][lane * NR + c] + quarter[1][lane * NR + c]) + (quarter[2][lane * NR + c] + quarter[3][lane * NR + c]);
  const long gi = x % prm.m, gj = x / prm.m;
  R* dst = prm.c + (gi + gj * prm.ldc) * NR;
  const R* cin = prm.cin + (gi + gj * prm.ldcin) * NR;
  if constexpr (!T::CPLX) {
    R v = prm.alpha * acc[0];
    if (prm.accumulate) v += dst[0];
    if (prm.beta != R(0)) v += prm.beta * cin[0];
    dst[0] = v;
  } else {
    const R ar = prm.alpha, ai = prm.alpha_im, br = prm.beta, bi = prm.beta_im;
    R vr = ar * acc[0] - ai * acc[1], vi = ar * acc[1] + ai * acc[0];
    if (prm.accumulate) {
      vr += dst[0];
      vi += dst[1];
    }
    if (br != R(0) || bi != R(0)) {
      const R cr = cin[0], ci = cin[1];
      vr += br * cr - bi * ci;
      vi += br * ci + bi * cr;
    }
    dst[0] = vr;
    dst[1] = vi;
  }
}

// Persistent batch: items (problem, tile row, tile column), the first gridDim.x dealt out by
// workgroup, the others taken from *counter (zero at launch) as workgroups become free. The next
// item is drawn while a tile runs. Every workgroup ends once its item is past the list. 64 x 64
// tiles, a quarter of the inner dimension per wave: a group of a dozen problems of some hundred rows
// fills the CUs, which its 128 x 128 tiles did not, and its longest tile takes an eighth of the time.
// 1024^3 problems back to back: 62.5 TFLOP/s (128 x 128 tiles, three workgroups per CU: 57.1). Calls
// on page-locked memory, bound by the host link and its copy commands: 48 problems of 64 to 1024
// rows and columns 2776 -> 2339 us, 12 of 64 to 1400 1357 -> 747, 200 of 64 to 3000 41.3 -> 37.8 ms.
template <typename T, bool A_KC, bool B_KC, int WBM, int WBN, int S>
__global__ __launch_bounds__(256, 2) void gemm_ks_batched_kernel(const GemmParams<typename T::R>* __restrict__ probs,
                                                                 const int* __restrict__ items, int n_items,
                                                                 int* __restrict__ counter) {
  __shared__ int next;
  int it = blockIdx.x;
  while (it < n_items) {
    int drawn = 0;
    if (threadIdx.x == 0) drawn = atomicAdd(counter, 1);
    const GemmParams<typename T::R> prm = probs[items[3 * it]];
    tile_at<T, A_KC, B_KC, WBM, WBN, S>(prm, prm.opa == 'C', prm.opb == 'C', items[3 * it + 1] * 16 * WBM,
                                        items[3 * it + 2] * 16 * WBN);
    if (threadIdx.x == 0) next = drawn;
    __syncthreads();  // `next` is there, and every wave is done with the tile's LDS
    it = (int)gridDim.x + __builtin_amdgcn_readfirstlane(next);
    // the next tile's barriers stand between this read and the next write of `next`
  }
}

// ---------------------------------------------------------------------------------------------
// Launches of one element type
// ---------------------------------------------------------------------------------------------
template <typename T, int WBM, int WBN, int S>
hipError_t launch_shape(const GemmParams<typename T::R>& p, hipStream_t s) {
  const dim3 grid((unsigned)ks_tiles(KsShape{WBM, WBN}, p.m, p.n)), block(256);
  const bool akc = p.opa != 'N', bkc = p.opb == 'N';
  if (akc && bkc) hipLaunchKernelGGL((gemm_ks_kernel<T, true, true, WBM, WBN, S>), grid, block, 0, s, p);
  else if (akc) hipLaunchKernelGGL((gemm_ks_kernel<T, true, false, WBM, WBN, S>), grid, block, 0, s, p);
  else if (bkc) hipLaunchKernelGGL((gemm_ks_kernel<T, false, true, WBM, WBN, S>), grid, block, 0, s, p);
  else hipLaunchKernelGGL((gemm_ks_kernel<T, false, false, WBM, WBN, S>), grid, block, 0, s, p);
  return hipGetLastError();
}

template <typename T, int WBM, int WBN, int S>
hipError_t launch_group(const GemmParams<typename T::R>* tiles, int count, hipStream_t s) {
  TileGroup<typename T::R> g;
  int wg = 0;
  if (!make_group(tiles, count, 16 * WBM, 16 * WBN, g, wg)) return hipErrorInvalidValue;
  const dim3 grid(wg), block(256);
  const bool akc = g.base.opa != 'N', bkc = g.base.opb == 'N';
  if (akc && bkc) hipLaunchKernelGGL((gemm_ks_group_kernel<T, true, true, WBM, WBN, S>), grid, block, 0, s, g);
  else if (akc) hipLaunchKernelGGL((gemm_ks_group_kernel<T, true, false, WBM, WBN, S>), grid, block, 0, s, g);
  else if (bkc) hipLaunchKernelGGL((gemm_ks_group_kernel<T, false, true, WBM, WBN, S>), grid, block, 0, s, g);
  else hipLaunchKernelGGL((gemm_ks_group_kernel<T, false, false, WBM, WBN, S>), grid, block, 0, s, g);
  return hipGetLastError();
}

template <typename T, int WBM, int WBN, int S>
hipError_t launch_split(const GemmParams<typename T::R>& p, int parts, void* ws, hipStream_t s) {
  const long tiles = ks_tiles(KsShape{WBM, WBN}, p.m, p.n);
  if (parts < 2 || tiles * parts > kSplitMaxWorkgroups) return hipErrorInvalidValue;
  const dim3 grid((unsigned)(tiles * parts)), block(256);
  const bool akc = p.opa != 'N', bkc = p.opb == 'N';
  typename T::R* sums = (typename T::R*)ws;
  if (akc && bkc) hipLaunchKernelGGL((gemm_ks_split_kernel<T, true, true, WBM, WBN, S>), grid, block, 0, s, p, parts, sums);
  else if (akc) hipLaunchKernelGGL((gemm_ks_split_kernel<T, true, false, WBM, WBN, S>), grid, block, 0, s, p, parts, sums);
  else if (bkc) hipLaunchKernelGGL((gemm_ks_split_kernel<T, false, true, WBM, WBN, S>), grid, block, 0, s, p, parts, sums);
  else hipLaunchKernelGGL((gemm_ks_split_kernel<T, false, false, WBM, WBN, S>), grid, block, 0, s, p, parts, sums);
  const dim3 sum_grid((unsigned)(((long)p.m * p.n + 63) / 64));
  hipLaunchKernelGGL((split_sum_kernel<T>), sum_grid, block, 0, s, p, parts, sums);
  return hipGetLastError();
}

}  // namespace ks
}  // namespace tmm
