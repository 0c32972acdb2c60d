// Ozaki-style split-precision DGEMM on INT8 matrix cores (gfx950).
//
// Scheme (Ozaki, Ogita, Oishi, Rump 2012, "Error-free transformations of matrix multiplication
// by using fast routines of matrix multiplication and its applications", in the integer-MMU form
// of Ootomo, Ozaki, Yokota 2024):
//   * every row i of op(A) is scaled by 2^-ea[i] (ea[i] = exponent with max_k |a_ik| < 2^ea[i]),
//     every column j of op(B) by 2^-eb[j]; the scaled values lie in (-1, 1);
//   * each scaled value is cut into s slices of 7 bits: x = sum_p S_p 2^(-7p) + r, S_p in
//     [-127, 127] (int8), |r| < 2^(-7s); the cut is exact in FP64 (scaling by powers of two and
//     removing integer parts);
//   * C = alpha * 2^(ea[i]+eb[j]) * sum_{p+q <= s+1} 2^(-7(p+q)) (S^A_p S^B_q)_ij + beta * C,
//     where every slice product runs on v_mfma_i32_16x16x64_i8 with exact int32 accumulation:
//     one product is bounded by k*127^2, so a launch sums only as many products of one diagonal
//     d = p+q as keep d_count*k*127^2 < 2^31;
//   * each launch adds its exact int32 sum, converted to FP64 and scaled by the power of two,
//     into C (the alpha/beta epilogue is fused into the first launch of a C tile).
// FP64 is used only for the exponent extraction, the slicing, and the recombination/epilogue.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <cmath>
#include <mutex>

#include "tmm_crt_loop.inc"
#include "tmm_kernels.h"
#include "tmm_ozaki.h"

namespace tmm {
namespace {

typedef int32_t i32x4 __attribute__((ext_vector_type(4)));
constexpr int kExpNone = -100000;  // row without a nonzero entry

__device__ __forceinline__ int frexp_exp_of(double v) {
  // exponent e with |v| < 2^e (frexp convention), kExpNone for 0; subnormals get -1022
  const uint64_t bits = __double_as_longlong(v) & 0x7FFFFFFFFFFFFFFFull;
  if (bits == 0) return kExpNone;
  const int be = (int)(bits >> 52);
  return be == 0 ? -1022 : be - 1022;
}

// ---------------------------------------------------------------------------------------------
// Exponents: e[r] = max over k of frexp-exponent(|x(r, k)|). x(r, k) at p[k + r*ld] (KC) or
// p[r + k*ld] (RC). A workgroup of 1024 threads takes a few rows over the whole inner dimension, so
// every e[r] has one writer: no initialising launch and no atomics. Many loads of a thread are in
// flight together (8 per batch). Bound by memory: two operands of 4096 x 4096 65 us (4.1 TB/s), of
// 2048 x 2048 14 us; with atomics, one load at a time and 64 workgroups, one row-contiguous operand
// of 2048 x 2048 took 108 us.
// ---------------------------------------------------------------------------------------------
struct OperandSrc {
  const double* p;
  long ld;
  int kc, rows, k;
  int* e;     // rows exponents
  int* flag;  // behind them: non-zero if an entry is non-finite or at least 2^kFallbackExp
};

// 16 rows per workgroup, 128 contiguous bytes of a row-contiguous operand (4, to spread few rows over
// more CUs, ran slower: 500 x 40000 twice, 171 us against 140).
constexpr int kExpRows = 16;

__device__ __forceinline__ void exponents16(const OperandSrc& o, int block, int* lds) {
  const int r0 = block * kExpRows, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int m = kExpNone;
  if (o.kc) {  // a wave per row
    const int r = r0 + wave;
    if (r < o.rows) {
      const double* row = o.p + (long)r * o.ld;
#pragma unroll 8
      for (int kk = lane; kk < o.k; kk += 64) m = max(m, frexp_exp_of(row[kk]));
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) m = max(m, __shfl_xor(m, off));
    if (lane == 0 && r < o.rows) o.e[r] = m;
    return;
  }
  const int r = r0 + (lane & 15);  // 16 rows of 4 k per wave and load
  if (r < o.rows) {
    const double* q = o.p + r;
#pragma unroll 8
    for (int kk = threadIdx.x >> 4; kk < o.k; kk += 64) m = max(m, frexp_exp_of(q[(long)kk * o.ld]));
  }
  m = max(m, __shfl_xor(m, 16));
  m = max(m, __shfl_xor(m, 32));
  if (lane < 16) lds[wave * 16 + lane] = m;
  __syncthreads();
  if (threadIdx.x < 16 && r < o.rows) {
    for (int w = 1; w < 16; ++w) m = max(m, lds[w * 16 + lane]);
    o.e[r] = m;
  }
}

// Exponents of two operands, the second's workgroups behind the first's. A grid holds fewer than 2^32 threads in one
// dimension, which 2^26 rows exceed: from kExpGridX workgroups on they go on in the second one.
constexpr int kExpGridX = 1 << 20;
__global__ __launch_bounds__(1024) void exponents_kernel(OperandSrc a, OperandSrc b) {
  __shared__ int lds[256];
  const int w = (int)(blockIdx.y * gridDim.x + blockIdx.x);
  const int na = (a.rows + kExpRows - 1) / kExpRows, nb = (b.rows + kExpRows - 1) / kExpRows;
  if (w < na) exponents16(a, w, lds);
  else if (w - na < nb) exponents16(b, w - na, lds);
}

// *flag from the operand's exponents, by one workgroup. Inf and NaN have frexp-exponent 1025, so an
// exponent above kFallbackExp marks the operand for the native fallback.
__device__ __forceinline__ void operand_flag(const OperandSrc& o) {
  int big = 0;
  for (int r = threadIdx.x; r < o.rows; r += blockDim.x) big |= o.e[r] > kFallbackExp;
  big = __syncthreads_or(big);
  if (threadIdx.x == 0) *o.flag = big ? 1 : 0;
}

__global__ __launch_bounds__(1024) void operand_flag_kernel(OperandSrc a, OperandSrc b) {
  if (blockIdx.x == 0) operand_flag(a);
  else operand_flag(b);
}

// ---------------------------------------------------------------------------------------------
// Slicing: S[p][r][k] (int8, row stride kpad, slice stride rows_pad*kpad) for r < rows_pad,
// k < kpad; zero outside the matrix. Each thread cuts 4 consecutive k of one row.
// ---------------------------------------------------------------------------------------------
template <bool KC>
__global__ __launch_bounds__(256) void split_kernel(const double* __restrict__ p, long ld, int rows, int k,
                                                    const int* __restrict__ e, int nslices, int rows_pad, int kpad,
                                                    int8_t* __restrict__ s) {
  const long tid = (long)blockIdx.x * 256 + threadIdx.x;
  const int k4 = kpad / 4;
  int r, kq;
  if (KC) {  // consecutive threads walk k of one row
    r = (int)(tid / k4);
    kq = (int)(tid % k4);
  } else {  // consecutive threads walk rows at one k
    r = (int)(tid % rows_pad);
    kq = (int)(tid / rows_pad);
  }
  if (r >= rows_pad || kq >= k4) return;
  double x[4];
  int sg[4];
  const int er = r < rows ? e[r] : kExpNone;
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int kk = kq * 4 + t;
    double v = 0.0;
    if (r < rows && kk < k) v = KC ? p[(long)kk + (long)r * ld] : p[(long)r + (long)kk * ld];
    sg[t] = v < 0.0 ? -1 : 1;
    // |v| * 2^-er in [0, 1): exact (power-of-two scaling)
    x[t] = er == kExpNone ? 0.0 : ldexp(fabs(v), -er);
  }
  const long plane = (long)rows_pad * kpad;
  int8_t* out = s + (long)r * kpad + (long)kq * 4;
  for (int q = 0; q < nslices; ++q) {
    uint32_t word = 0;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const double y = x[t] * 128.0;  // exact
      const double d = floor(y);       // 0..127
      x[t] = y - d;                    // exact
      const int v = sg[t] * (int)d;
      word |= ((uint32_t)(uint8_t)(int8_t)v) << (8 * t);
    }
    *(uint32_t*)(out + q * plane) = word;
  }
}

// ---------------------------------------------------------------------------------------------
// INT8 slice-product GEMM with FP64 scaled accumulation.
// WG tile 256x256, 4 waves (2x2) of 128x128 = 8x8 blocks of 16x16, k-step 64 per stage, one
// workgroup per CU. Operands go global -> LDS with global_load_lds_dwordx4 into an OZ_S-stage
// ring (OZ_S - 1 stages in flight while the MFMAs of one run): with one wave per SIMD nothing
// else hides the load latency, so a register-staged double buffer left the MFMAs idle most of
// each stage.
//
// Stage layout per operand: [row][slot][16 bytes], 64 bytes per row. The slices are k-contiguous
// with rows padded to 256 and k to 64, so every load is in bounds and unguarded. A wave
// instruction fills 16 consecutive rows (1 KB, lane l at byte 16*l): lanes 4j..4j+3 read the
// 64 contiguous bytes of row j, lane l landing in slot l % 4, which receives the k-chunk
// (l % 4) ^ oz_swz(row). The MFMA fragment read of one k-chunk by 16 consecutive rows then hits
// 8 distinct 16-byte bank groups per 8 lanes (rows r, r+1 share a swizzle and lie 64 bytes
// apart): no bank conflicts.
// ---------------------------------------------------------------------------------------------
// Residue products of nmod moduli: planes a + q*a_plane and b + q*b_plane (int8, k-step tiled
// layout: one contiguous 16 KB block per 256 rows and 64 k, blocks of a row block in k order, 64-byte
// rows inside) into res + q*plane (uint8 in [0, modulus) at i + j*ldres; ldres a multiple of 16,
// rows m..ldres-1 receive padding). The launch does nothing if *fa | *fb is non-zero (the operands'
// fallback flags, an entry is non-finite or at least 2^kFallbackExp in magnitude).
struct CrtProductParams {
  int m, n, kpad, nmod;
  const int8_t* a;
  long a_plane;
  const int8_t* b;
  long b_plane;
  uint8_t* res;
  long plane, ldres;
  const int* fa;
  const int* fb;
  int magic[kCrtMaxModuli];       // ceil(2^38 / m)
  unsigned neg_m[kCrtMaxModuli];  // -m
};

constexpr int OZ_BM = 256, OZ_BN = 256, OZ_BK = 64;
constexpr int OZ_S = 4;                         // LDS ring stages
constexpr int OZ_TILE = OZ_BM * OZ_BK;          // bytes of one operand stage (16 KB)
constexpr int OZ_STAGE = 2 * OZ_TILE;           // A and B
constexpr int OZ_LOADS = OZ_TILE / (16 * 256);  // 16-byte loads per thread per operand and stage
static_assert(OZ_BM == OZ_BN && OZ_LOADS == 4, "load mapping assumes square 256x256 tiles, k-step 64");

__device__ __forceinline__ int oz_swz(int r) { return (r >> 1) & 3; }

// s_waitcnt immediate: vmcnt(vm) with lgkmcnt(0), expcnt not waited (gfx9 encoding: vmcnt bits
// [3:0] and [15:14], expcnt [6:4], lgkmcnt [11:8]).
template <int VM>
__device__ __forceinline__ void wait_vm_lgkm0() {
  static_assert(VM >= 0 && VM < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((VM & 15) | ((VM >> 4) << 14) | (7 << 4));
}

// Issue this wave's loads of one operand stage: OZ_LOADS instructions of 16 rows x 64 bytes.
__device__ __forceinline__ void oz_issue(const int8_t* __restrict__ base, long row_stride, int row0, int k0,
                                         int8_t* stage, int wave, int lane) {
#pragma unroll
  for (int t = 0; t < OZ_LOADS; ++t) {
    const int inst = wave * OZ_LOADS + t;  // 0..15
    const int local = inst * 16 + (lane >> 2);
    const int q = (lane & 3) ^ oz_swz(local);
    const int8_t* src = base + (long)(row0 + local) * row_stride + k0 + 16 * q;
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                     (__attribute__((address_space(3))) void*)(stage + inst * 1024), 16, 0, 0);
  }
}

__device__ __forceinline__ i32x4 oz_frag(const int8_t* stage, int row, int g) {
  return *(const i32x4*)(stage + row * 64 + ((g ^ oz_swz(row)) << 4));
}

// Output tile t of an nbm x nbn grid, walked in groups of 4 tile-rows column by column (the ~32
// tiles an XCD runs at once then share A and B strips in its L2).
__device__ __forceinline__ void oz_tile(int t, int nbm, int nbn, int& m0, int& n0) {
  const int GROUP_M = 4, in_group = GROUP_M * nbn, group = t / in_group, first_m = group * GROUP_M;
  const int gsz = min(nbm - first_m, GROUP_M), rr = t - group * in_group;
  m0 = (first_m + rr % gsz) * OZ_BM;
  n0 = (rr / gsz) * OZ_BN;
}

// Item w of n, XCD-aware: workgroup w runs on XCD w % 8, so each XCD gets a contiguous range.
__device__ __forceinline__ int xcd_range(int w, int n) {
  if (n < 32) return w;
  const int xcd = w % 8, per = n / 8, rem = n % 8;
  return xcd * per + min(xcd, rem) + w / 8;
}

// Residues of four sums as the bytes of a word: each congruent to its sum mod m and in [0, m], for
// |sum| <= 2^30 and 129 <= m <= 256. h = sum M / 2^32 with M = ceil(2^38 / m), q = h / 2^6: sum M / 2^38
// differs from sum / m by less than 2^30 / 2^38 < 1 / m (not at all for 256), so q is the floored
// quotient, or one less where a negative sum is a multiple of m (the residue is then m, as good as 0
// for the reconstruction). Of sum - q m only the low byte is needed, so that part runs on pairs of 16
// bits. 17 instructions for four sums with the reads of the accumulators; with one wave per SIMD an
// instruction takes 5.5 cycles and a conversion between integers and floats 8.5, and the FP32 form
// (fold to 21 bits, convert, fma, floor, fma, convert and pack) took 36 of them, a quarter of the
// kernel's time at an inner dimension of 2048.
__device__ __forceinline__ unsigned residues_of_sums(const i32x4& sum, int magic, unsigned neg_m) {
  typedef unsigned short us2 __attribute__((ext_vector_type(2)));
  const us2 factor = {(unsigned short)neg_m, (unsigned short)neg_m};
  unsigned r[2];
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const int s0 = sum[2 * p], s1 = sum[2 * p + 1];
    // the low halves of two words
    const unsigned h = __builtin_amdgcn_perm((unsigned)__mulhi(s1, magic), (unsigned)__mulhi(s0, magic), 0x05040100u);
    const unsigned s = __builtin_amdgcn_perm((unsigned)s1, (unsigned)s0, 0x05040100u);
    const us2 q = __builtin_bit_cast(us2, h) >> (unsigned short)6;
    r[p] = __builtin_bit_cast(unsigned, (us2)(q * factor + __builtin_bit_cast(us2, s)));
  }
  return __builtin_amdgcn_perm(r[1], r[0], 0x06040200u);
}

// Residue epilogue of the product kernel: res[i + j*ldres] = acc mod m for the workgroup's
// 256x256 tile. The lane holds C(i = m0 + wm*128 + bi*16 + 4*lg + r, j = n0 + wn*128 + bj*16 + li) in
// acc[bj][bi][r] (B is the loop's first operand), so the four residues of an accumulator are
// consecutive rows: one word. The words go through the (then idle) LDS ring as a column-major
// tile with a 272-byte column stride (a wave's 64 words fall into 64 banks), then out as 16
// consecutive rows of a column per lane (16 lanes write one column's 256 bytes). ldres is a multiple
// of 16 and every row m0..m0+255 below ldres may be written (rows >= m hold padding).
constexpr int OZ_RES_STRIDE = 272;

__device__ __forceinline__ void oz_store_residues(const CrtProductParams& prm, int q, const i32x4 (&acc)[8][8], int m0,
                                                  int n0, int wm, int wn, int li, int lg, int8_t* lds) {
  const int magic = prm.magic[q];
  const unsigned neg_m = prm.neg_m[q];
  uint8_t* T = (uint8_t*)lds;
  __syncthreads();  // every wave is done with the ring
#pragma unroll
  for (int bj = 0; bj < 8; ++bj)
#pragma unroll
    for (int bi = 0; bi < 8; ++bi) {
      const unsigned w = residues_of_sums(acc[bj][bi], magic, neg_m);
      *(unsigned*)(T + (wn * 128 + bj * 16 + li) * OZ_RES_STRIDE + wm * 128 + bi * 16 + 4 * lg) = w;
    }
  __syncthreads();
  uint8_t* res = prm.res + (long)q * prm.plane;
  const long rows_left = prm.ldres - m0;  // rows of the plane from m0 on (a multiple of 16)
#pragma unroll 4
  for (int x = 0; x < 16; ++x) {
    const int c = (int)threadIdx.x + 256 * x, col = c >> 4, ch = c & 15;
    if (n0 + col >= prm.n || 16 * ch >= rows_left) continue;
    const uint4 v = *(const uint4*)(T + col * OZ_RES_STRIDE + 16 * ch);
    *(uint4*)(res + (long)(m0 + 16 * ch) + (long)(n0 + col) * prm.ldres) = v;
  }
}

__global__ __launch_bounds__(256, 1) void ozaki_gemm_kernel(OzakiGemmParams prm) {
  __shared__ __attribute__((aligned(16))) int8_t lds[OZ_S * OZ_STAGE];  // 128 KB
  if (prm.fa && (*prm.fa | *prm.fb)) return;  // the native fallback computes this product

  int m0, n0;
  const int nbm = (prm.m + OZ_BM - 1) / OZ_BM, nbn = (prm.n + OZ_BN - 1) / OZ_BN;
  oz_tile(xcd_range(blockIdx.x, nbm * nbn), nbm, nbn, m0, n0);

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave & 1, wn = wave >> 1;
  const int li = lane & 15, lg = lane >> 4;

  i32x4 acc[8][8];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[i][j] = i32x4{0, 0, 0, 0};

  // slice indices packed into 4-bit fields of two scalars, so the loop reads no kernel argument
  // memory (a scalar load in flight would make the compiler wait for every LDS read at once)
  unsigned long long pa_bits = 0, pb_bits = 0;
  for (int q = 0; q < prm.nprod; ++q) {
    pa_bits |= (unsigned long long)prm.pa[q] << (4 * q);
    pb_bits |= (unsigned long long)prm.pb[q] << (4 * q);
  }
  const int kt0 = prm.k_begin / OZ_BK;
  const int nkt = (prm.k_end - prm.k_begin) / OZ_BK;
  const int total = nkt * prm.nprod;
  // stage `it` = slice pair it / nkt at k-tile kt0 + it % nkt, into ring slot `slot`
  auto issue = [&](int it, int slot) {
    int8_t* st = lds + slot * OZ_STAGE;
    const int pr = it / nkt, k0 = (kt0 + it % nkt) * OZ_BK;
    oz_issue(prm.a + (long)((pa_bits >> (4 * pr)) & 15) * prm.a_slice_stride, prm.kpad, m0, k0, st, wave, lane);
    oz_issue(prm.b + (long)((pb_bits >> (4 * pr)) & 15) * prm.b_slice_stride, prm.kpad, n0, k0, st + OZ_TILE, wave,
             lane);
  };

  // wait until this wave's loads of stage s have landed, given that `later` further stages are
  // also issued (2 * OZ_LOADS loads each), then the barrier
  auto wait_stage = [&](int later) {
    if (later >= 3) wait_vm_lgkm0<6 * OZ_LOADS>();
    else if (later == 2) wait_vm_lgkm0<4 * OZ_LOADS>();
    else if (later == 1) wait_vm_lgkm0<2 * OZ_LOADS>();
    else wait_vm_lgkm0<0>();
    __builtin_amdgcn_s_barrier();
  };

  auto frag_a = [&](int it, int i) {
    return oz_frag(lds + (it % OZ_S) * OZ_STAGE, wm * 128 + i * 16 + li, lg);
  };
  auto frag_b = [&](int it, int j) {
    return oz_frag(lds + (it % OZ_S) * OZ_STAGE + OZ_TILE, wn * 128 + j * 16 + li, lg);
  };

  // One barrier per stage. Every iteration issues exactly one stage of loads: past the end it
  // reloads the last stage into the slot just freed (never read again), so (OZ_S - 2) stages are
  // always in flight behind the awaited one and the waits need no tail cases.
  // Measured alternatives, on 8192^3 with 4 slice products (MI355X): this loop 1.74 POPS; reading
  // the next stage's fragments across a mid-stage barrier 1.54 (the register allocator then
  // shuffles the 256 accumulator registers); two 256x128 workgroups per CU 1.54 (LDS-bound); the
  // register-staged double buffer 1.27.
  if (total > 0) {
#pragma unroll
    for (int s = 0; s < OZ_S - 1; ++s) issue(min(s, total - 1), s);
  }
  for (int it = 0; it < total; ++it) {
    // stage it has landed for every wave and every wave's reads of stage it-1 are done: that
    // slot takes stage it+OZ_S-1
    wait_stage(OZ_S - 2);
    issue(min(it + OZ_S - 1, total - 1), (it + OZ_S - 1) % OZ_S);
    // the fragment reads first, in the order the MFMAs consume them
    i32x4 af[8], bf[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) af[i] = frag_a(it, i);
#pragma unroll
    for (int j = 0; j < 8; ++j) bf[j] = frag_b(it, j);
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int i = 0; i < 8; ++i) acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(bf[j], af[i], acc[i][j], 0, 0, 0);
    __builtin_amdgcn_sched_group_barrier(0x100, 16, 0);  // DS reads
    __builtin_amdgcn_sched_group_barrier(0x008, 64, 0);  // then the MFMAs
  }
  // no LDS load may still be landing when the workgroup ends (its LDS is handed to the next one)
  wait_vm_lgkm0<0>();

  // lane holds C(i = m0 + wm*128 + bi*16 + li, j = n0 + wn*128 + bj*16 + 4*lg + r)
  // epilogue: C = alpha * 2^(ea+eb+shift) * acc + (accumulate ? C : 0) + beta * C_in
#pragma unroll
  for (int bi = 0; bi < 8; ++bi) {
    const int gi = m0 + wm * 128 + bi * 16 + li;
    if (gi >= prm.m) continue;
    const int ei = prm.ea[gi];
#pragma unroll
    for (int bj = 0; bj < 8; ++bj) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int gj = n0 + wn * 128 + bj * 16 + 4 * lg + r;
        if (gj >= prm.n) continue;
        const int ej = prm.eb[gj];
        double v = 0.0;
        if (ei != kExpNone && ej != kExpNone) v = ldexp(prm.alpha * (double)acc[bi][bj][r], ei + ej + prm.shift);
        double* dst = prm.c + (long)gi + (long)gj * prm.ldc;
        if (prm.accumulate) v += *dst;
        if (prm.beta != 0.0) v += prm.beta * prm.cin[(long)gi + (long)gj * prm.ldcin];
        *dst = v;
      }
    }
  }
}

// Residue products of all moduli in one launch, with the main loop scheduled by hand: the tile,
// ring slot layout, load mapping and fragment layout of ozaki_gemm_kernel, operands in k-step tiled
// layout, a 4-stage ring (128 KB of LDS) and the k-step schedule of gen_crt_loop.py (fragments
// double-buffered in registers, loads and LDS reads interleaved with the MFMAs, one barrier
// half-way through each k-step). B is the loop's first operand (see oz_store_residues). A 5-stage
// ring (160 KB) gave the same rate.
// A k-step takes 1090 to 1140 cycles, 1024 of them MFMAs, and a tile some 22000 cycles more (first
// loads, residues, 64 KB of stores, the next workgroup's start; 26000 before the residues ran on
// integers). What bounds a long inner dimension is power: the clock falls from 2.7 GHz at 64 to 2.0 at
// 2048 and 1.85 at 8192. 2048 x 2048 x k, 16 moduli, in us: k = 64 42.3 -> 34.3, 512 61.4 -> 59.0, 2048
// 122.2 -> 117.4.
__global__ __launch_bounds__(256, 1) void crt_product_kernel(CrtProductParams prm) {
  constexpr int S = 4;  // the generated loop's ring
  __shared__ __attribute__((aligned(16))) int8_t lds[S * OZ_STAGE];
  if (*prm.fa | *prm.fb) return;  // the native fallback computes this product

  // items modulus by modulus, so that the XCDs' ranges share few residue planes
  const int nbm = (prm.m + OZ_BM - 1) / OZ_BM, nbn = (prm.n + OZ_BN - 1) / OZ_BN, ntiles = nbm * nbn;
  const int item = xcd_range(blockIdx.x, prm.nmod * ntiles), q = item / ntiles;
  int m0, n0;
  oz_tile(item - q * ntiles, nbm, nbn, m0, n0);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave & 1, wn = wave >> 1;
  const int li = lane & 15, lg = lane >> 4;

  i32x4 acc[8][8];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[i][j] = i32x4{0, 0, 0, 0};

  const int nkt = prm.kpad / OZ_BK;
  {
    const unsigned lds0 = (unsigned)(uintptr_t)((__attribute__((address_space(3))) int8_t*)lds);
    // load t of a k-step fills LDS rows (4*wave + t)*16 .. +15 of each operand (the oz_issue mapping)
    const unsigned ldsw = __builtin_amdgcn_readfirstlane(lds0 + (unsigned)wave * 4 * 1024);
    // k-step tiled operands: row `local` of a 16 KB k-step block at byte local*64, load t covers
    // rows (4*wave + t)*16 + lane/4, i.e. the bytes at vo[t] (the swizzle depends on lane/4)
    unsigned vo[4];
#pragma unroll
    for (int t = 0; t < 4; ++t)
      vo[t] = ((unsigned)(wave * 4 + t) * 16 + (lane >> 2)) * 64 + 16u * (unsigned)((lane & 3) ^ oz_swz(lane >> 2));
    // fragment reads (oz_frag): row w*128 + i*16 + li at byte row*64 + 16*(lg ^ swz(row)); the
    // swizzle depends on li only, so fragment i sits at a fixed offset i*1024 from the lane base
    const unsigned lane_off = (unsigned)li * 64 + ((unsigned)(lg ^ oz_swz(li)) << 4);
    unsigned ra[S], rb[S];
#pragma unroll
    for (int s = 0; s < S; ++s) {
      ra[s] = lds0 + s * OZ_STAGE + wn * 8192 + lane_off;
      rb[s] = lds0 + s * OZ_STAGE + OZ_TILE + wm * 8192 + lane_off;
    }
    const int8_t* gA = prm.b + (long)q * prm.b_plane + (long)(n0 / OZ_BN) * nkt * OZ_TILE;
    const int8_t* gB = prm.a + (long)q * prm.a_plane + (long)(m0 / OZ_BM) * nkt * OZ_TILE;
    unsigned cnt = (unsigned)nkt, adv = (unsigned)nkt - 1, tmp, tmp2;
    i32x4 fa[8], fb[8], ga[8], gb[8];
    // M0 is written by the loop (LDS DMA destination); nothing else in this kernel uses it
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
    asm volatile(TMM_CRT_LOOP_S4 : TMM_CRT_OUTPUTS : TMM_CRT_INPUTS_S4 : "memory", "m0", "scc");
#pragma clang diagnostic pop
  }
  oz_store_residues(prm, q, acc, m0, n0, wm, wn, li, lg, lds);
}

}  // namespace

// ---------------------------------------------------------------------------------------------
// Scratch of the no-allocation entry point. In host code `scratch` names a host-side stand-in,
// not device memory: only its per-device address from hipGetSymbolAddress is ever handed to a
// kernel or a copy. Nothing in it has to start at zero (every kernel of the emulation writes what
// it later reads), and calls that overlap on one device share it.
// ---------------------------------------------------------------------------------------------
static __device__ __align__(256) char scratch[kOzakiScratchBytes];

namespace {
constexpr int kScratchDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kScratchDevices] = {};
}  // namespace

hipError_t ozaki_scratch_resolve() {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kScratchDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (g_scratch_ptr[dev]) return hipSuccess;
  void* p = nullptr;
  e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (e != hipSuccess) return e;
  g_scratch_ptr[dev] = p;
  return hipSuccess;
}

void* ozaki_scratch(int device) {
  if (device < 0 || device >= kScratchDevices) return nullptr;
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  return g_scratch_ptr[device];
}

namespace {
// Exponents of `count` (1 or 2) operands, in one launch.
hipError_t launch_exponents(const OperandSrc* o, int count, hipStream_t s) {
  OperandSrc none{};
  const OperandSrc& b = count > 1 ? o[1] : none;
  const int blocks = (o[0].rows + kExpRows - 1) / kExpRows + (b.rows + kExpRows - 1) / kExpRows;
  if (blocks > 0) {
    const dim3 grid(std::min(blocks, kExpGridX), (blocks + kExpGridX - 1) / kExpGridX);
    hipLaunchKernelGGL(exponents_kernel, grid, dim3(1024), 0, s, o[0], b);
  }
  return hipGetLastError();
}
}  // namespace

hipError_t ozaki_split(const double* p, long ld, bool kc, int rows, int k, const int* e, int nslices, int rows_pad,
                       int kpad, int8_t* out, hipStream_t s) {
  const long threads = (long)rows_pad * (kpad / 4);
  if (threads == 0) return hipSuccess;
  const dim3 grid((unsigned)((threads + 255) / 256));
  if (kc) hipLaunchKernelGGL(split_kernel<true>, grid, dim3(256), 0, s, p, ld, rows, k, e, nslices, rows_pad, kpad, out);
  else hipLaunchKernelGGL(split_kernel<false>, grid, dim3(256), 0, s, p, ld, rows, k, e, nslices, rows_pad, kpad, out);
  return hipGetLastError();
}

hipError_t ozaki_gemm(const OzakiGemmParams& p, hipStream_t s) {
  if (p.m <= 0 || p.n <= 0) return hipSuccess;
  const int nbm = (p.m + OZ_BM - 1) / OZ_BM, nbn = (p.n + OZ_BN - 1) / OZ_BN;
  hipLaunchKernelGGL(ozaki_gemm_kernel, dim3(nbm * nbn), dim3(256), 0, s, p);
  return hipGetLastError();
}

namespace {
inline long pad_to(long x, long q) { return (x + q - 1) / q * q; }
inline size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }
}  // namespace

// exponents of `rows` rows followed by the operand's fallback flag
static inline size_t exp_flag_bytes(int rows) { return align256((size_t)std::max(rows, 1) * 4 + 4); }

size_t ozaki_workspace_bytes(int m, int n, int k, int nslices) {
  const long kpad = pad_to(std::max(k, 1), OZ_BK), mpad = pad_to(m, OZ_BM), npad = pad_to(n, OZ_BN);
  return exp_flag_bytes(m) + exp_flag_bytes(n) + align256((size_t)nslices * mpad * kpad) +
         align256((size_t)nslices * npad * kpad);
}

namespace {
// The native FP64 kernel on the original operands, doing its work only when fa or fb is set.
hipError_t native_fallback(char opa, char opb, int m, int n, int k, double alpha, const double* a, long lda,
                           const double* b, long ldb, double beta, const double* cin, long ldcin, bool accumulate,
                           double* c, long ldc, const int* fa, const int* fb, hipStream_t s) {
  GemmParams<double> p;
  p.opa = opa;
  p.opb = opb;
  p.m = m;
  p.n = n;
  p.k = k;
  p.alpha = alpha;
  p.alpha_im = 0.0;
  p.a = a;
  p.lda = lda;
  p.b = b;
  p.ldb = ldb;
  p.beta = beta;
  p.beta_im = 0.0;
  p.cin = cin;
  p.ldcin = ldcin;
  p.accumulate = accumulate ? 1 : 0;
  p.c = c;
  p.ldc = ldc;
  p.variant = 1;
  p.gate_a = fa;
  p.gate_b = fb;
  return launch_gemm_d(p, s);
}
}  // namespace

hipError_t ozaki_dgemm(char opa, char opb, int m, int n, int k, double alpha, const double* a, long lda,
                       const double* b, long ldb, double beta, const double* cin, long ldcin, bool accumulate,
                       double* c, long ldc, int nslices, void* work, hipStream_t s, int* n_products) {
  if (n_products) *n_products = 0;
  if (m <= 0 || n <= 0) return hipSuccess;
  if (nslices < 1 || nslices > 12) return hipErrorInvalidValue;
  const long kpad = pad_to(std::max(k, 1), OZ_BK), mpad = pad_to(m, OZ_BM), npad = pad_to(n, OZ_BN);
  char* w = (char*)work;
  int* ea = (int*)w;
  w += exp_flag_bytes(m);
  int* eb = (int*)w;
  w += exp_flag_bytes(n);
  int* fa = ea + m;  // fallback flags
  int* fb = eb + n;
  int8_t* sa = (int8_t*)w;
  w += align256((size_t)nslices * mpad * kpad);
  int8_t* sb = (int8_t*)w;
  // op(A) rows: k-contiguous when A is transposed; op(B) columns: k-contiguous when B is not.
  const bool a_kc = opa != 'N', b_kc = opb == 'N';
  hipError_t e;
  const OperandSrc src[2] = {{a, lda, a_kc, m, k, ea, fa}, {b, ldb, b_kc, n, k, eb, fb}};
  if ((e = launch_exponents(src, 2, s)) != hipSuccess) return e;
  hipLaunchKernelGGL(operand_flag_kernel, dim3(2), dim3(1024), 0, s, src[0], src[1]);
  if ((e = ozaki_split(a, lda, a_kc, m, k, ea, nslices, (int)mpad, (int)kpad, sa, s)) != hipSuccess) return e;
  if ((e = ozaki_split(b, ldb, b_kc, n, k, eb, nslices, (int)npad, (int)kpad, sb, s)) != hipSuccess) return e;

  // products of one diagonal d = p+q share the power-of-two scale; a launch sums at most
  // gmax of them so the int32 accumulation stays exact: gmax * k * 127^2 < 2^31.
  const long per_product = (long)std::max(k, 1) * 127 * 127;
  const int gmax = (int)std::max<long>(1, std::min<long>(kOzakiMaxProducts, 2147483647L / per_product));
  // with k > 2^31/127^2 a single product could overflow: process k in ranges
  const long krange = per_product > 2147483647L ? pad_to(2147483647L / (127 * 127) - OZ_BK, OZ_BK) : kpad;
  OzakiGemmParams P{};
  P.m = m;
  P.n = n;
  P.kpad = (int)kpad;
  P.a = sa;
  P.a_slice_stride = mpad * kpad;
  P.b = sb;
  P.b_slice_stride = npad * kpad;
  P.ea = ea;
  P.eb = eb;
  P.fa = fa;
  P.fb = fb;
  P.alpha = alpha;
  P.c = c;
  P.ldc = ldc;
  bool first = true;
  int count = 0;
  for (long k0 = 0; k0 < kpad; k0 += krange) {
    P.k_begin = (int)k0;
    P.k_end = (int)std::min(kpad, k0 + krange);
    for (int d = 2; d <= nslices + 1; ++d) {
      int np = 0;
      for (int p = 1; p <= nslices; ++p) {
        const int q = d - p;
        if (q < 1 || q > nslices) continue;
        P.pa[np] = p - 1;
        P.pb[np] = q - 1;
        ++np;
        if (np == gmax || p == nslices || d - p - 1 < 1) {
          P.nprod = np;
          P.shift = -7 * d;
          P.accumulate = first ? (accumulate ? 1 : 0) : 1;
          P.beta = first ? beta : 0.0;
          P.cin = cin;
          P.ldcin = ldcin;
          if ((e = ozaki_gemm(P, s)) != hipSuccess) return e;
          first = false;
          count += np;
          np = 0;
        }
      }
    }
  }
  if ((e = native_fallback(opa, opb, m, n, k, alpha, a, lda, b, ldb, beta, cin, ldcin, accumulate, c, ldc, fa, fb,
                           s)) != hipSuccess)
    return e;
  if (n_products) *n_products = count;
  return hipSuccess;
}


// =============================================================================================
// Ozaki scheme II: integer products modulo pairwise coprime moduli, CRT reconstruction.
//
// (Ozaki, Uchino, Imamura 2025, "Ozaki Scheme II: A GEMM-oriented emulation of floating-point
// matrix multiplication using an integer modular technique".)
//   * a'(i,k) = round(|a(i,k)| * 2^(bits - ea[i])) * sign, |a'| <= 2^bits, likewise b'(k,j) with
//     eb[j]; op(A)op(B) = 2^(ea[i] + eb[j] - 2 bits) * (A'B')(i,j) up to the rounding of the inputs
//     (at most 2^-bits of the row / column maximum per entry);
//   * |(A'B')(i,j)| <= k 2^(2 bits) < M/4 with M the product of the moduli, so A'B' is fixed by its
//     residues r_t = A'B' mod m_t; each residue comes from one INT8 product of the balanced
//     residues of A' and B' (entries in [-128, 127], exact int32 sums for k <= 65536);
//   * CRT sum: A'B' = sum_t r_t W_t - q M with W_t = (M/m_t) y_t, y_t = (M/m_t)^-1 mod m_t, and
//     q = rint(sum_t r_t y_t / m_t) (in FP64 within 2^-35 of sum_t r_t W_t / M, whose distance to
//     the integer q is |A'B'| / M < 1/4, so the rounding is never in doubt); the sum is taken
//     exactly in 26-bit FP64 limbs (every partial sum an integer below 2^40), carried into
//     non-negative limbs and added from the top in double-double: exact when A'B' is
//     representable, otherwise within one unit in the last place.
// =============================================================================================
namespace {

constexpr int kCrtModuli[kCrtMaxModuli] = {256, 255, 253, 251, 247, 241, 239, 233, 229, 227,
                                           223, 211, 199, 197, 193, 191, 181, 179, 173, 167};
static_assert(kCrtModuli[kCrtMaxModuli - 1] >= 129, "residues_of_sums: 2^38 / m fits a signed factor");

constexpr long inv_mod(long a, long m) {  // extended Euclid; a and m coprime
  long g = m, x = 0, x1 = 1, a1 = a % m;
  while (a1 != 0) {
    const long q = g / a1, t = g - q * a1;
    g = a1;
    a1 = t;
    const long tx = x - q * x1;
    x = x1;
    x1 = tx;
  }
  return ((x % m) + m) % m;
}

// Constants of the CRT sum for the first N moduli, fixed by the moduli list and known at compile
// time (the unrolled loops take them as scalar operands): f[t] = y_t / m_t rounded to FP64, the
// 26-bit limbs of W_t = (M/m_t) y_t and of M (M <= 256^N needs L = ceil(8N/26) limbs).
constexpr int kLimbBits = 26;
template <int N>
struct CrtSum {
  static constexpr int L = (8 * N + kLimbBits - 1) / kLimbBits;
  double f[N];
  double w[N][L];
  double mm[L];
};

// x *= s for a little-endian number of L 26-bit limbs (s <= 256; the product fits the L limbs)
template <int L>
constexpr void limbs_mul_small(unsigned long long (&x)[L], unsigned long long s) {
  unsigned long long carry = 0;
  for (int i = 0; i < L; ++i) {
    const unsigned long long v = x[i] * s + carry;
    x[i] = v & ((1ull << kLimbBits) - 1);
    carry = v >> kLimbBits;
  }
}

template <int N>
constexpr CrtSum<N> make_crt_sum() {
  constexpr int L = CrtSum<N>::L;
  CrtSum<N> d{};
  unsigned long long M[L] = {};
  M[0] = 1;
  for (int t = 0; t < N; ++t) limbs_mul_small<L>(M, (unsigned long long)kCrtModuli[t]);
  for (int i = 0; i < L; ++i) d.mm[i] = (double)M[i];
  for (int t = 0; t < N; ++t) {
    const long m = kCrtModuli[t];
    long mt_mod = 1;  // (M / m_t) mod m_t
    for (int s = 0; s < N; ++s)
      if (s != t) mt_mod = mt_mod * kCrtModuli[s] % m;
    const long y = inv_mod(mt_mod, m);
    unsigned long long W[L] = {};
    W[0] = (unsigned long long)y;
    for (int s = 0; s < N; ++s)
      if (s != t) limbs_mul_small<L>(W, (unsigned long long)kCrtModuli[s]);
    for (int i = 0; i < L; ++i) d.w[t][i] = (double)W[i];
    d.f[t] = (double)y / (double)m;
  }
  return d;
}

template <int N>
struct CrtSumTable {
  static constexpr CrtSum<N> v = make_crt_sum<N>();
};

// Constants of the operands' residues, per modulus: 2^30 mod m (balanced), 1 / m, m.
struct ResidueConsts {
  int n;
  double c30[kCrtMaxModuli], inv[kCrtMaxModuli], m[kCrtMaxModuli];
};

ResidueConsts residue_consts(int n) {
  ResidueConsts c{};
  c.n = n;
  for (int t = 0; t < n; ++t) {
    const int m = kCrtModuli[t], r = (1 << 30) % m;
    c.c30[t] = r > m / 2 ? r - m : r;
    c.inv[t] = 1.0 / m;
    c.m[t] = m;
  }
  return c;
}

// Byte offset of entry (r, k) in a residue plane of rows_pad x kpad in k-step tiled layout: one
// contiguous 16 KB block per (256-row block, 64-k step), blocks of a row block in k order, rows of
// 64 bytes inside a block. A k-step of a 256-row product tile is then one contiguous 16 KB read.
__device__ __forceinline__ long crt_tiled_offset(int r, int k, int kpad) {
  return ((long)(r >> 8) * (kpad >> 6) + (k >> 6)) * 16384 + (r & 255) * 64 + (k & 63);
}

// Balanced residues of an operand's scaled, rounded entries x = rint(v 2^(bits - e)), |x| <= 2^62: one
// int8 plane per modulus, rows_pad x kpad in k-step tiled layout (zero outside the matrix). A
// workgroup takes 64 rows x 64 k through LDS (global reads of 512 contiguous bytes either way; its
// 64 rows fill 4 KB of one 16 KB block per plane), then each thread 16 consecutive k of one row.
//   x = xh 2^30 + xl exactly (|xh| <= 2^32, |xl| <= 2^29); y = xh c30 + xl is congruent to x, an exact
//   integer below 2^40; q = rint(y / m) by adding and taking off 1.5 2^52: y times the rounded 1 / m
//   is off by less than 2^-20, and y / m lies at least 1 / (2m) from a half for odd m and is exact
//   for 256, so y - q m is the balanced residue (128 and -128 are the same byte); adding 1.5 2^52
//   once more leaves it in the low byte. Five FP64 instructions and 3/4 of a byte permutation, all
//   full-rate; an integer form needs a wider reduction. Bound by memory once the loads of a tile are in
//   flight together and nothing waits on them one by one: 16 moduli of two operands of 1000 x 1000 16
//   us, of 2048 x 2048 41 us (4.9 TB/s), of 4096 x 4096 188 us; with a bounds check around every load
//   and LDS read 20, 46 and 227 us; a launch per operand with the integer form took 87 us at 2048 x
//   2048.
struct ResidueDst {
  int bits, kpad;
  long plane;
  int8_t* out;
};
constexpr int kResStride = 65;  // doubles per LDS row (odd: 64 rows of one k fall into distinct banks)

__device__ __forceinline__ void residues64(const OperandSrc& o, const ResidueDst& d, const ResidueConsts& cc, int block,
                                           int q0, int q1, double* tile) {
  const int t = threadIdx.x, nks = d.kpad / 64;
  const int r0 = (((block >> 2) / nks) * 4 + (block & 3)) * 64, k0 = (block >> 2) % nks * 64;
  // all 16 loads in flight, out-of-range ones from the last row and k, before any goes to LDS
  double v[16] = {};
  if (o.rows > 0 && o.k > 0) {
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const int hi = (t >> 6) + 4 * j, lo = t & 63;
      const int r = min(r0 + (o.kc ? hi : lo), o.rows - 1), kk = min(k0 + (o.kc ? lo : hi), o.k - 1);
      v[j] = o.p[o.kc ? (long)kk + (long)r * o.ld : (long)r + (long)kk * o.ld];
    }
  }
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const int hi = (t >> 6) + 4 * j, lo = t & 63;
    const int rl = o.kc ? hi : lo, kl = o.kc ? lo : hi;
    tile[rl * kResStride + kl] = r0 + rl < o.rows && k0 + kl < o.k ? v[j] : 0.0;
  }
  __syncthreads();
  // 4 lanes take a row: a wave's 64 stores of 16 bytes fill 1 KB
  const int rl = t >> 2, g = t & 3, r = r0 + rl;
  const int er = r < o.rows ? o.e[r] : kExpNone;
  const int shift = er == kExpNone ? 0 : d.bits - er;  // a row without an exponent holds zeros
  double xh[16], xl[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const double x = rint(ldexp(tile[rl * kResStride + 16 * g + i], shift));
    xh[i] = rint(x * 0x1p-30);
    xl[i] = fma(-xh[i], 0x1p30, x);
  }
  const double magic = 0x1.8p52;
  int8_t* out = d.out + crt_tiled_offset(r, k0 + 16 * g, d.kpad);
  double c30_next = cc.c30[q0], inv_next = cc.inv[q0], m_next = cc.m[q0];
  for (int q = q0; q < q1; ++q) {
    const double c30 = c30_next, inv = inv_next, m = m_next;
    const int qn = min(q + 1, q1 - 1);  // the next modulus's constants come in under this one's work
    c30_next = cc.c30[qn];
    inv_next = cc.inv[qn];
    m_next = cc.m[qn];
    unsigned b[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const double y = fma(xh[i], c30, xl[i]);
      const double n = fma(y, inv, magic) - magic;
      b[i] = (unsigned)__double2loint(fma(-n, m, y) + magic);
    }
    unsigned w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      // bytes 0 of two words into the low and, shifted, the high half
      const unsigned lo = __builtin_amdgcn_perm(b[4 * i + 1], b[4 * i], 0x0c0c0400);
      const unsigned hi = __builtin_amdgcn_perm(b[4 * i + 3], b[4 * i + 2], 0x04000c0c);
      w[i] = lo | hi;
    }
    *(uint4*)(out + q * d.plane) = uint4{w[0], w[1], w[2], w[3]};
  }
}

// Residues of two operands, the second's workgroups behind the first's (na), and their fallback
// flags; the moduli dealt out over blockIdx.y.
__global__ __launch_bounds__(256) void residues_kernel(OperandSrc a, ResidueDst da, int na, OperandSrc b, ResidueDst db,
                                                       ResidueConsts cc) {
  __shared__ double tile[64 * kResStride];
  const int w = blockIdx.x, part = blockIdx.y, parts = gridDim.y;
  const int q0 = cc.n * part / parts, q1 = cc.n * (part + 1) / parts;
  if (w < na) {
    if (w == 0 && part == 0) operand_flag(a);
    residues64(a, da, cc, w, q0, q1, tile);
  } else {
    if (w == na && part == 0) operand_flag(b);
    residues64(b, db, cc, w - na, q0, q1, tile);
  }
}

// S_i -> [0, 2^26) for every limb but the top, the carries moving up (each step exact: the limbs
// are integers below 2^40 and floor of a power-of-two scaling is exact).
template <int L>
__device__ __forceinline__ void crt_carry(double* S) {
#pragma unroll
  for (int i = 0; i < L - 1; ++i) {
    const double c = floor(S[i] * 0x1p-26);
    S[i] = fma(-c, 0x1p26, S[i]);
    S[i + 1] = S[i + 1] + c;
  }
}

// FP64 value of Y = sum_i S_i 2^(26 i) (exact integer limbs, |Y| < M/4): carried, made
// non-negative (the sign is the top limb's once the others lie in [0, 2^26)), paired into limbs
// below 2^52 and added from the top in double-double. Exact when Y is representable, as every
// top-down partial sum then is; otherwise within one unit in the last place. Contraction is off
// so that each line is one IEEE operation (tests/crt_model.py mirrors them).
template <int L>
__device__ __forceinline__ double crt_limbs_value(double* S) {
#pragma clang fp contract(off)
  crt_carry<L>(S);
  const double sgn = S[L - 1] < 0.0 ? -1.0 : 1.0;
#pragma unroll
  for (int i = 0; i < L; ++i) S[i] = sgn * S[i];
  crt_carry<L>(S);
  constexpr int NP = (L + 1) / 2;
  double P[NP];
#pragma unroll
  for (int j = 0; j < NP; ++j) P[j] = 2 * j + 1 < L ? fma(S[2 * j + 1], 0x1p26, S[2 * j]) : S[2 * j];
  double h = ldexp(P[NP - 1], 52 * (NP - 1)), lo = 0.0;
#pragma unroll
  for (int j = NP - 2; j >= 0; --j) {
    const double T = ldexp(P[j], 52 * j);
    const double s = h + T;  // TwoSum(h, T) = s + e exactly
    const double bb = s - h;
    const double e = (h - (s - bb)) + (T - bb);
    h = s;
    lo = lo + e;
  }
  return sgn * (h + lo);
}

// C(i,j) = alpha * 2^(ea[i] + eb[j] - 2 bits) * CRT(residues) + (accumulate ? C : 0) + beta*C_in.
// A thread takes 4 consecutive rows of one column: the residues of the 4 sit in one 32-bit word
// per plane (ldres is a multiple of 16), and each constant of the sum serves the 4 rows in turn.
// Grid: x over row quads, y over columns (strided).
template <int N>
__global__ __launch_bounds__(256) void crt_reconstruct_kernel(const uint8_t* __restrict__ res, long plane, long ldres,
                                                              int m, int n, const int* __restrict__ ea,
                                                              const int* __restrict__ eb, int bits,
                                                              double alpha, double beta, const double* __restrict__ cin,
                                                              long ldcin, int accumulate, double* __restrict__ c,
                                                              long ldc, const int* __restrict__ fa,
                                                              const int* __restrict__ fb) {
  constexpr int L = CrtSum<N>::L;
  constexpr CrtSum<N> D = CrtSumTable<N>::v;
  if (*fa | *fb) return;  // the native fallback writes this C
  const int i0 = 4 * (blockIdx.x * 256 + threadIdx.x);
  if (i0 >= m) return;
  int ei[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) ei[u] = i0 + u < m ? ea[i0 + u] : kExpNone;
  for (int j = blockIdx.y; j < n; j += gridDim.y) {
    const long off = (long)i0 + (long)j * ldres;
    uint32_t w[N];
#pragma unroll
    for (int t = 0; t < N; ++t) w[t] = *(const uint32_t*)(res + off + (long)t * plane);
    const int ej = eb[j];
    // per row: the q sum sum_t r_t f_t and the limb sums sum_t r_t W_ti (exact integers)
    double qs[4] = {0.0, 0.0, 0.0, 0.0}, S[4][L];
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int i = 0; i < L; ++i) S[u][i] = 0.0;
#pragma unroll
    for (int t = 0; t < N; ++t) {
      double r[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) r[u] = (double)((w[t] >> (8 * u)) & 255u);
#pragma unroll
      for (int u = 0; u < 4; ++u) qs[u] = fma(r[u], D.f[t], qs[u]);
#pragma unroll
      for (int i = 0; i < L; ++i)
#pragma unroll
        for (int u = 0; u < 4; ++u) S[u][i] = fma(r[u], D.w[t][i], S[u][i]);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (i0 + u >= m) break;
      const double q = rint(qs[u]);
#pragma unroll
      for (int i = 0; i < L; ++i) S[u][i] = fma(-q, D.mm[i], S[u][i]);
      const double y = crt_limbs_value<L>(S[u]);
      double out = 0.0;
      if (ei[u] != kExpNone && ej != kExpNone) out = alpha * ldexp(y, ei[u] + ej - 2 * bits);
      const int i = i0 + u;
      double* dst = c + (long)i + (long)j * ldc;
      if (accumulate) out += *dst;
      if (beta != 0.0) out += beta * cin[(long)i + (long)j * ldcin];
      *dst = out;
    }
  }
}

template <int N>
void launch_reconstruct(dim3 grid, hipStream_t s, const uint8_t* res, long plane, long ldres, int m, int n,
                        const int* ea, const int* eb, int bits, double alpha, double beta,
                        const double* cin, long ldcin, int accumulate, double* c, long ldc) {
  // the fallback flags follow the exponents of each prepared operand
  hipLaunchKernelGGL(crt_reconstruct_kernel<N>, grid, dim3(256), 0, s, res, plane, ldres, m, n, ea, eb, bits, alpha,
                     beta, cin, ldcin, accumulate, c, ldc, ea + m, eb + n);
}

}  // namespace

int ozaki2_bits(int nmod, int k) {
  double l = 0;
  for (int t = 0; t < nmod && t < kCrtMaxModuli; ++t) l += std::log2((double)kCrtModuli[t]);
  const int lk = (int)std::ceil(std::log2((double)std::max(k, 1)));
  // k * 2^(2 bits) <= 2^(l - 2) < M / 4
  const int bits = (int)std::floor((l - 2.0 - lk) / 2.0);
  return std::max(1, std::min(62, bits));
}

size_t ozaki2_operand_bytes(int rows, int k, int nmod) {
  const long kr = pad_to(std::max(k, 1), OZ_BK), rows_pad = pad_to(std::max(rows, 1), OZ_BM);
  return exp_flag_bytes(rows) + align256((size_t)nmod * rows_pad * kr);
}

size_t ozaki2_product_bytes(int m, int n, int nmod) {
  return align256((size_t)nmod * pad_to(std::max(m, 1), 16) * std::max(n, 1));
}

size_t ozaki2_workspace_bytes(int m, int n, int k, int nmod) {
  const int kr = std::min(std::max(k, 1), kCrtMaxK);
  return ozaki2_operand_bytes(m, kr, nmod) + ozaki2_operand_bytes(n, kr, nmod) + ozaki2_product_bytes(m, n, nmod);
}

namespace {
struct PrepareJob {
  const double* p;
  long ld;
  bool kc;
  int rows;
  void* out;
};
// Prepare `count` (1 or 2) operands of inner dimension k: their exponents in one launch, their
// residues and flags in another.
hipError_t prepare(const PrepareJob* jobs, int count, int k, int nmod, hipStream_t s) {
  const int kp = (int)pad_to(std::max(k, 1), OZ_BK), bits = ozaki2_bits(nmod, k);
  OperandSrc src[2] = {};
  ResidueDst dst[2] = {};
  int blocks[2] = {0, 0};
  for (int i = 0; i < count; ++i) {
    const PrepareJob& j = jobs[i];
    const long rows_pad = pad_to(j.rows, OZ_BM);
    int* e = (int*)j.out;
    src[i] = OperandSrc{j.p, j.ld, j.kc, j.rows, k, e, e + j.rows};
    dst[i] = ResidueDst{bits, kp, rows_pad * kp, (int8_t*)j.out + exp_flag_bytes(j.rows)};
    blocks[i] = (int)(rows_pad / 64 * (kp / 64));
  }
  const hipError_t e = launch_exponents(src, count, s);
  if (e != hipSuccess) return e;
  // Up to about one workgroup per CU the moduli go to two sets of them, which read the operands twice
  // but keep more waves in flight: whole emulated products of 500^3 (128 workgroups) 40.7 -> 38.9 us,
  // 700^3 (264) 45.6 -> 44.5; 850^3 (448) 52.8 -> 54.4, 2048^3 216 -> 224; four sets gain nothing more.
  const int all = blocks[0] + blocks[1], parts = all <= 288 ? 2 : 1;
  hipLaunchKernelGGL(residues_kernel, dim3(all, parts), dim3(256), 0, s, src[0], dst[0], blocks[0], src[1], dst[1],
                     residue_consts(nmod));
  return hipGetLastError();
}
}  // namespace

hipError_t ozaki2_prepare(const double* p, long ld, bool kc, int rows, int k, int nmod, void* out, hipStream_t s) {
  if (rows <= 0) return hipSuccess;
  if (nmod < kCrtMinModuli || nmod > kCrtMaxModuli || k > kCrtMaxK) return hipErrorInvalidValue;
  const PrepareJob job{p, ld, kc, rows, out};
  return prepare(&job, 1, k, nmod, s);
}

hipError_t ozaki2_products(int m, int n, int k, const void* pa, const void* pb, int nmod, void* work, hipStream_t s) {
  if (m <= 0 || n <= 0) return hipSuccess;
  if (nmod < kCrtMinModuli || nmod > kCrtMaxModuli || k > kCrtMaxK) return hipErrorInvalidValue;
  const int kp = (int)pad_to(std::max(k, 1), OZ_BK);
  const long mpad = pad_to(m, OZ_BM), npad = pad_to(n, OZ_BN);
  const int8_t* ra = (const int8_t*)pa + exp_flag_bytes(m);
  const int8_t* rb = (const int8_t*)pb + exp_flag_bytes(n);
  CrtProductParams P{};
  P.m = m;
  P.n = n;
  P.kpad = kp;
  P.nmod = nmod;
  P.a = ra;
  P.a_plane = mpad * kp;
  P.b = rb;
  P.b_plane = npad * kp;
  P.res = (uint8_t*)work;
  P.ldres = pad_to(m, 16);
  P.plane = P.ldres * n;
  P.fa = (const int*)pa + m;  // operands with a fallback flag skip the products
  P.fb = (const int*)pb + n;
  auto constants = [&P](int at, int modulus) {
    P.magic[at] = (int)(((1L << 38) + modulus - 1) / modulus);
    P.neg_m[at] = (unsigned)-modulus;
  };
  const long ntiles = (mpad / OZ_BM) * (npad / OZ_BN);
  // All moduli in one launch while a modulus has few tiles: alone it leaves CUs idle (2048^3: 64
  // tiles on 256 CUs, 16 launches 425 us) or its last round does. From 1024 tiles on that is below
  // 5%, and one launch per modulus keeps the XCDs on the same operand strips (16384 x 16384 x 8192:
  // 28.6 ms against 30.1 for one launch; 8192^3: 8.0 against 8.3; 4096^3, 256 tiles: 1.49 against
  // 1.40).
  if (ntiles < 1024) {
    for (int t = 0; t < nmod; ++t) constants(t, kCrtModuli[t]);
    hipLaunchKernelGGL(crt_product_kernel, dim3((unsigned)(ntiles * nmod)), dim3(256), 0, s, P);
    return hipGetLastError();
  }
  P.nmod = 1;
  for (int t = 0; t < nmod; ++t) {
    constants(0, kCrtModuli[t]);
    hipLaunchKernelGGL(crt_product_kernel, dim3((unsigned)ntiles), dim3(256), 0, s, P);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    P.a += P.a_plane;
    P.b += P.b_plane;
    P.res += P.plane;
  }
  return hipSuccess;
}

hipError_t ozaki2_reconstruct(int m, int n, int k, double alpha, const void* pa, const void* pb, double beta,
                              const double* cin, long ldcin, bool accumulate, double* c, long ldc, int nmod,
                              const void* work, hipStream_t s) {
  if (m <= 0 || n <= 0) return hipSuccess;
  if (nmod < kCrtMinModuli || nmod > kCrtMaxModuli || k > kCrtMaxK) return hipErrorInvalidValue;
  const int* ea = (const int*)pa;
  const int* eb = (const int*)pb;
  const uint8_t* rc = (const uint8_t*)work;
  const int bits = ozaki2_bits(nmod, k);
  const long ldres = pad_to(m, 16), plane = ldres * n;
  const dim3 grid((unsigned)((m + 1023) / 1024), (unsigned)std::min(n, 32768));
  const int acc = accumulate ? 1 : 0;
  switch (nmod) {
#define TMM_CRT_CASE(NN) \
  case NN:                                                                                                     \
    launch_reconstruct<NN>(grid, s, rc, plane, ldres, m, n, ea, eb, bits, alpha, beta, cin, ldcin, acc, c, ldc); \
    break;
    TMM_CRT_CASE(6) TMM_CRT_CASE(7) TMM_CRT_CASE(8) TMM_CRT_CASE(9) TMM_CRT_CASE(10) TMM_CRT_CASE(11)
    TMM_CRT_CASE(12) TMM_CRT_CASE(13) TMM_CRT_CASE(14) TMM_CRT_CASE(15) TMM_CRT_CASE(16) TMM_CRT_CASE(17)
    TMM_CRT_CASE(18) TMM_CRT_CASE(19) TMM_CRT_CASE(20)
#undef TMM_CRT_CASE
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t ozaki2_fallback(char opa, char opb, int m, int n, int k, double alpha, const double* a, long lda,
                           const double* b, long ldb, double beta, const double* cin, long ldcin, bool accumulate,
                           double* c, long ldc, const void* pa, const void* pb, hipStream_t s) {
  if (m <= 0 || n <= 0) return hipSuccess;
  return native_fallback(opa, opb, m, n, k, alpha, a, lda, b, ldb, beta, cin, ldcin, accumulate, c, ldc,
                         (const int*)pa + m, (const int*)pb + n, s);
}

hipError_t ozaki2_product(int m, int n, int k, double alpha, const void* pa, const void* pb, double beta,
                          const double* cin, long ldcin, bool accumulate, double* c, long ldc, int nmod, void* work,
                          hipStream_t s) {
  const hipError_t e = ozaki2_products(m, n, k, pa, pb, nmod, work, s);
  if (e != hipSuccess) return e;
  return ozaki2_reconstruct(m, n, k, alpha, pa, pb, beta, cin, ldcin, accumulate, c, ldc, nmod, work, s);
}

hipError_t ozaki2_dgemm(char opa, char opb, int m, int n, int k, double alpha, const double* a, long lda,
                        const double* b, long ldb, double beta, const double* cin, long ldcin, bool accumulate,
                        double* c, long ldc, int nmod, void* work, hipStream_t s, int* n_products) {
  if (n_products) *n_products = 0;
  if (m <= 0 || n <= 0) return hipSuccess;
  if (nmod < kCrtMinModuli || nmod > kCrtMaxModuli) return hipErrorInvalidValue;
  const int kr = std::min(std::max(k, 1), kCrtMaxK);
  char* pa = (char*)work;
  char* pb = pa + ozaki2_operand_bytes(m, kr, nmod);
  char* rc = pb + ozaki2_operand_bytes(n, kr, nmod);
  const bool a_kc = opa != 'N', b_kc = opb == 'N';
  hipError_t e;
  int count = 0;
  const int nranges = (std::max(k, 1) + kCrtMaxK - 1) / kCrtMaxK;
  for (int q = 0; q < nranges; ++q) {
    // one pass per k range of at most kCrtMaxK: exponents and residues of both operands, nmod
    // INT8 products and a reconstruction that adds into C (alpha/beta/accumulate on the first
    // pass only)
    const int k0 = q * kCrtMaxK, kk = std::min(k, k0 + kCrtMaxK) - k0;
    const double* ap = a + (a_kc ? (long)k0 : (long)k0 * lda);
    const double* bp = b + (b_kc ? (long)k0 : (long)k0 * ldb);
    const PrepareJob jobs[2] = {{ap, lda, a_kc, m, pa}, {bp, ldb, b_kc, n, pb}};
    if ((e = prepare(jobs, 2, kk, nmod, s)) != hipSuccess) return e;
    if ((e = ozaki2_product(m, n, kk, alpha, pa, pb, q == 0 ? beta : 0.0, cin, ldcin, q == 0 ? accumulate : true, c,
                            ldc, nmod, rc, s)) != hipSuccess)
      return e;
    if ((e = ozaki2_fallback(opa, opb, m, n, kk, alpha, ap, lda, bp, ldb, q == 0 ? beta : 0.0, cin, ldcin,
                             q == 0 ? accumulate : true, c, ldc, pa, pb, s)) != hipSuccess)
      return e;
    count += nmod;
  }
  if (n_products) *n_products = count;
  return hipSuccess;
}

}  // namespace tmm
