// SELL-64 storage and kernels for scalar sparse operators.
//
// Rows are grouped in slices of 64 (one wavefront).  Inside a slice the k-th
// entry of every row is stored contiguously (column-major), so each lane
// streams its own row while the wavefront's loads stay fully coalesced: 64
// consecutive columns (256 B) and values (512 B in FP64) per step.  One thread
// owns one row and sums it in the stored (ColumnStencil) order, so with
// EXACT = true the row sums reproduce the reference's sequential loops bit for
// bit (SparseBlockMatrix::vmult, src/LinAlg/sparseblockmatrix.xx:378-392;
// MgInterpolatorMatrix::restrict_zero / prolongate_add,
// src/Discretization/Q1/mginterpolatormatrix.cc:123-147).  Reduced-precision
// (non-exact) sweeps over levels of few slices may instead split a slice over
// K wavefronts (k_sell_split); exact sweeps of long rows form the products in
// several wavefronts and fold them in the stored order (k_sell_fold).  A slice
// whose rows share pattern and values reads one row of values (kSharedBit).
#pragma once

#include <type_traits>

#include "gh_kernels.h"

namespace gh {

// ------------------------------------------------------------------ ops
// init(row) gives the accumulator start, step folds one entry, finish writes.
template <typename T, bool EXACT>
__device__ __forceinline__ T fma_step(T acc, T a, T x) {
  if constexpr (EXACT) return add_rn(acc, mul_rn(a, x));
  else return acc + a * x;
}
template <typename T, bool EXACT>
__device__ __forceinline__ T fms_step(T acc, T a, T x) {
  if constexpr (EXACT) return add_rn(acc, -mul_rn(a, x));
  else return acc - a * x;
}

template <typename Y, typename T, bool EXACT>
struct SpmvOp {  // y = d * (A x) + b * y
  static constexpr bool kExact = EXACT;
  Y* y;
  T d, b;
  bool read_y;
  __device__ __forceinline__ T init(int64_t) const { return (T)0; }
  __device__ __forceinline__ T step(T acc, T a, T x) const { return fma_step<T, EXACT>(acc, a, x); }
  // the step of a product formed and rounded before (exact ops)
  __device__ __forceinline__ T fold(T acc, T p) const { return add_rn(acc, p); }
  static __device__ __forceinline__ T neutral() { return (T)-0.0; }  // fold(acc, neutral) = acc
  __device__ __forceinline__ void finish(int64_t r, T acc) const {
    T v = EXACT ? mul_rn(d, acc) : d * acc;
    if (read_y) v = EXACT ? add_rn(v, mul_rn(b, (T)y[r])) : v + b * (T)y[r];
    y[r] = (Y)v;
  }
};

template <typename T, bool EXACT>
struct ResidualOp {  // r = b - A x: r starts at b and subtracts each a_ij x_j in order
  static constexpr bool kExact = EXACT;
  T* r;
  const T* b;
  __device__ __forceinline__ T init(int64_t i) const { return b[i]; }
  __device__ __forceinline__ T step(T acc, T a, T x) const { return fms_step<T, EXACT>(acc, a, x); }
  __device__ __forceinline__ T fold(T acc, T p) const { return add_rn(acc, -p); }
  static __device__ __forceinline__ T neutral() { return (T)0.0; }
  __device__ __forceinline__ void finish(int64_t i, T acc) const { r[i] = acc; }
};

template <typename T, typename DT, bool EXACT>
struct JacobiOp {  // xn = x + omega * (dinv * (b - A x))
  static constexpr bool kExact = EXACT;
  T* xn;
  const T* x;
  const T* b;
  const DT* dinv;
  T omega;
  int richardson;
  __device__ __forceinline__ T init(int64_t i) const { return b[i]; }
  __device__ __forceinline__ T step(T acc, T a, T xx) const { return fms_step<T, EXACT>(acc, a, xx); }
  __device__ __forceinline__ T fold(T acc, T p) const { return add_rn(acc, -p); }
  static __device__ __forceinline__ T neutral() { return (T)0.0; }
  __device__ __forceinline__ void finish(int64_t i, T h) const {
    if (!richardson) h = EXACT ? mul_rn((T)dinv[i], h) : (T)dinv[i] * h;
    xn[i] = EXACT ? add_rn(x[i], mul_rn(omega, h)) : x[i] + omega * h;
  }
};

template <typename T>
struct RestrictOp {  // uc = R uf (packed weights)
  T* uc;
  __device__ __forceinline__ T init(int64_t) const { return (T)0; }
  __device__ __forceinline__ T step(T acc, T w, T x) const { return add_rn(acc, mul_rn(w, x)); }
  __device__ __forceinline__ void finish(int64_t i, T acc) const { uc[i] = acc; }
};

// uc = R uf, and the coarse level's first smoothing sweep from a zero start
// in the same pass: ux = 0 + omega * (dinv * (uc - 0)), the operations of a
// Jacobi (or Richardson) sweep whose iterate is zero
template <typename T, typename DT>
struct RestrictSmoothOp {
  T* uc;
  T* ux;
  const DT* dinv;
  T omega;
  int richardson;
  __device__ __forceinline__ T init(int64_t) const { return (T)0; }
  __device__ __forceinline__ T step(T acc, T w, T x) const { return add_rn(acc, mul_rn(w, x)); }
  __device__ __forceinline__ void finish(int64_t i, T acc) const {
    uc[i] = acc;
    T h = acc - (T)0;
    if (!richardson) h = (T)dinv[i] * h;
    ux[i] = (T)0 + omega * h;
  }
};

template <typename T>
struct ProlongAddOp {  // uf += P uc, term by term
  T* uf;
  __device__ __forceinline__ T init(int64_t i) const { return uf[i]; }
  __device__ __forceinline__ T step(T acc, T w, T x) const { return add_rn(acc, mul_rn(w, x)); }
  __device__ __forceinline__ void finish(int64_t i, T acc) const { uf[i] = acc; }
};

template <typename T, typename UT>
struct CorrectOp {  // v = P' uc ; u += mgomega * v  (empty rows leave u as it is)
  UT* u;
  T mgomega;
  __device__ __forceinline__ T init(int64_t) const { return (T)0; }
  __device__ __forceinline__ T step(T acc, T w, T x) const { return add_rn(acc, mul_rn(w, x)); }
  __device__ __forceinline__ void finish(int64_t i, T v) const {
    u[i] = (UT)add_rn((T)u[i], mul_rn(mgomega, v));
  }
};

// ---------------------------------------------------------------- kernels
// Workgroups are dealt to the 8 XCDs round-robin (workgroup i runs on XCD
// i mod 8).  Remapping the workgroup index gives every XCD one contiguous
// range of rows, so the x entries a row range gathers are fetched into that
// XCD's own L2 instead of into all eight.
constexpr unsigned kXcds = 8;
__device__ __forceinline__ unsigned xcd_block(unsigned b, unsigned G) {
  const unsigned q = G / kXcds, r = G % kXcds;
  const unsigned xcd = b % kXcds, k = b / kXcds;
  return xcd * q + (xcd < r ? xcd : r) + k;
}

// ------------------------------------------------- block matrices (BSell)
// B consecutive values of one x block, widened to the accumulator type;
// 16-byte vector loads where the data allow it (the host checks the alignment
// before it picks this kernel).
template <int B, typename T, typename Acc>
__device__ __forceinline__ void load_block_row(const T* __restrict__ p, Acc (&o)[B]) {
  if constexpr (B == 4 && std::is_same<T, double>::value) {
    typedef double d2 __attribute__((ext_vector_type(2)));
    const d2 a = *reinterpret_cast<const d2*>(p), b = *reinterpret_cast<const d2*>(p + 2);
    o[0] = (Acc)a.x; o[1] = (Acc)a.y; o[2] = (Acc)b.x; o[3] = (Acc)b.y;
  } else if constexpr (B == 4 && std::is_same<T, float>::value) {
    typedef float f4 __attribute__((ext_vector_type(4)));
    const f4 a = *reinterpret_cast<const f4*>(p);
    o[0] = (Acc)a.x; o[1] = (Acc)a.y; o[2] = (Acc)a.z; o[3] = (Acc)a.w;
  } else {
#pragma unroll
    for (int c = 0; c < B; ++c) o[c] = (Acc)ld(p + c);
  }
}

// One lane per component row t = i*B + r: for each kept block of row i (in
// the row's column order) sum = sum_c A(r, c) x_c from zero, then
// acc = op.step(acc, sum) -- the per-block sums of k_bsr, in the same order,
// so both kernels return the same bits.  Only all-zero block rows are left
// out (their sum is an exact zero).
template <int B, typename VT, typename XT, typename Acc, class Op>
__global__ __launch_bounds__(kBlock) void k_bsell(int64_t nslices, const uint32_t* __restrict__ sptr,
                                                  const int32_t* __restrict__ row,
                                                  const uint16_t* __restrict__ rlen,
                                                  const int32_t* __restrict__ col,
                                                  const VT* __restrict__ val,
                                                  const XT* __restrict__ x, Op op) {
  const int64_t g = (int64_t)xcd_block(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
  const int64_t s = g >> 6;
  if (s >= nslices) return;
  const int32_t t = row[g];
  if (t < 0) return;
  const int len = rlen[g];
  const int64_t p0 = (int64_t)sptr[s] * 64 + (threadIdx.x & 63);
  Acc acc = op.init(t);
  const int lane = threadIdx.x & 63;
  const int64_t v0 = (int64_t)sptr[s] * B * 64 + lane;  // value c of entry k: v0 + (k*B + c)*64
  int k = 0;
  // Four entries per step.  The step's value and x loads are all issued
  // before its arithmetic (the scheduling barrier keeps the compiler from
  // serialising the x gathers to save registers), and the next step's columns
  // are fetched one step ahead.
  int32_t c[4];
  if (len >= 4) {
#pragma unroll
    for (int u = 0; u < 4; ++u) c[u] = col[p0 + (int64_t)u * 64];
  }
  for (; k + 4 <= len; k += 4) {
    Acc m[4][B], q[4][B];
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int cc = 0; cc < B; ++cc) m[u][cc] = (Acc)ld(val + v0 + ((int64_t)(k + u) * B + cc) * 64);
#pragma unroll
    for (int u = 0; u < 4; ++u) load_block_row<B>(x + (int64_t)c[u] * B, q[u]);
    if (k + 8 <= len) {
#pragma unroll
      for (int u = 0; u < 4; ++u) c[u] = col[p0 + (int64_t)(k + 4 + u) * 64];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      Acc sum = (Acc)0;
#pragma unroll
      for (int cc = 0; cc < B; ++cc) sum = add_rn(sum, mul_rn(m[u][cc], q[u][cc]));
      acc = op.step(acc, sum);
    }
  }
  for (; k < len; ++k) {
    Acc m[B], q[B];
#pragma unroll
    for (int cc = 0; cc < B; ++cc) m[cc] = (Acc)ld(val + v0 + ((int64_t)k * B + cc) * 64);
    load_block_row<B>(x + (int64_t)col[p0 + (int64_t)k * 64] * B, q);
    Acc sum = (Acc)0;
#pragma unroll
    for (int cc = 0; cc < B; ++cc) sum = add_rn(sum, mul_rn(m[cc], q[cc]));
    acc = op.step(acc, sum);
  }
  op.finish(t, acc);
}

// k_bsell where one wavefront per slice is bound by the chain column -> x block
// of its longest rows (125 entries for a Stokes-LPS pressure row): a workgroup of
// kBSplit wavefronts takes a slice.  They form the per-block sums of kBSplit *
// kBEntries entries of the 64 rows at a time, side by side, into LDS, and
// wavefront 0 folds them into the rows in entry order.  Entry k of a round goes to
// wavefront k % kBSplit, so that the last, partial round is as short for each of
// them.  Entries past a row's end exist in the padded slice (column 0) and are
// formed but not folded.  Two buffers, one barrier per round.  Stokes-LPS
// residuals against k_bsell: 32^3 79 -> 33 us in FP64 (134 MB, 4.1 TB/s), 36 -> 22
// in FP32; 64^3 330 -> 251 (1.12 GB, 4.5 TB/s) and 182 -> 135; 4913 nodes 26 -> 13
// and 13 -> 10.4, launch and copy latency included.
constexpr int kBSplit = 4;
constexpr int kBEntries = 8;
template <int B, typename VT, typename XT, typename Acc, class Op>
__global__ __launch_bounds__(64 * kBSplit) void k_bsell_split(
    const uint32_t* __restrict__ sptr, const int32_t* __restrict__ row,
    const uint16_t* __restrict__ rlen, const int32_t* __restrict__ col,
    const VT* __restrict__ val, const XT* __restrict__ x, Op op) {
  constexpr int C = kBSplit * kBEntries;
  __shared__ Acc part[2][C][64];
  const int64_t s = xcd_block(blockIdx.x, gridDim.x);  // one slice per workgroup
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int64_t s0 = sptr[s];
  const int width = (int)(sptr[s + 1] - s0);
  const int32_t t = row[s * 64 + lane];  // -1: no row
  const int len = rlen[s * 64 + lane];
  const int32_t* cp = col + s0 * 64 + lane;
  const VT* vp = val + s0 * B * 64 + lane;
  Acc acc = (Acc)0;
  if (w == 0 && t >= 0) acc = op.init(t);
  // E entries from c0 on, every kBSplit-th from the wavefront's own; those past
  // the slice's width repeat its last one
  auto batch = [&](auto num, int c0, int buf) {
    constexpr int E = decltype(num)::value;
    Acc m[E][B], q[E][B];
    int32_t c[E];
    int64_t k[E];
#pragma unroll
    for (int u = 0; u < E; ++u) k[u] = min(c0 + u * kBSplit + w, width - 1);
#pragma unroll
    for (int u = 0; u < E; ++u) c[u] = cp[k[u] * 64];
#pragma unroll
    for (int u = 0; u < E; ++u)
#pragma unroll
      for (int cc = 0; cc < B; ++cc) m[u][cc] = (Acc)ld(vp + (k[u] * B + cc) * 64);
#pragma unroll
    for (int u = 0; u < E; ++u) load_block_row<B>(x + (int64_t)c[u] * B, q[u]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < E; ++u) {
      Acc sum = (Acc)0;
#pragma unroll
      for (int cc = 0; cc < B; ++cc) sum = add_rn(sum, mul_rn(m[u][cc], q[u][cc]));
      part[buf][u * kBSplit + w][lane] = sum;
    }
  };
  for (int c0 = 0, buf = 0; c0 < width; c0 += C, buf ^= 1) {
    // (the conditions are the same for the whole wavefront)
    const int left = width - c0 - w;
    if (left > 4 * kBSplit)
      batch(std::integral_constant<int, kBEntries>{}, c0, buf);
    else if (left > kBSplit)
      batch(std::integral_constant<int, 4>{}, c0, buf);
    else if (left > 0)
      batch(std::integral_constant<int, 1>{}, c0, buf);
    __syncthreads();
    if (w == 0) {
      const int n = min(C, width - c0);
#pragma unroll 8
      for (int u = 0; u < n; ++u) {
        const Acc sum = part[buf][u][lane];
        if (c0 + u < len) acc = op.step(acc, sum);
      }
    }
  }
  if (w == 0 && t >= 0) op.finish(t, acc);
}

// Which of the two runs.  The split pays where the chain of the longest rows is
// longer than the sweep's share of the chip takes: with few slices (2 per CU;
// 27-entry rows, B = 4, 500 slices 9.8 -> 6.5 us in FP64 and 5.1 -> 4.6 in FP32,
// 125 slices 7.4 -> 4.9 and 5.0 -> 3.9), and where a few long rows hold most of the
// entries (Stokes-LPS).  Otherwise the slices fill the chip one wavefront each, and
// LDS and barriers only cost: 9-entry rows (2D), 263 K nodes, B = 2 17 -> 25 us,
// B = 4 70 -> 94; 27-entry rows, 275 K nodes, B = 2 50 -> 58; 36 entries, 1000
// slices, B = 4 14.7 -> 16.7; 96 entries for every row, 2000 slices 36 -> 38.  Rows
// of up to 18 entries have too short a chain (13 entries, 16 slices 3.6 -> 3.9 us).
constexpr int kBSplitRow = 24, kBSplitLong = 64;
constexpr int64_t kBSplitSlices = 512;
inline bool bsell_is_split(const BSell& S) {
  if (S.width < kBSplitRow) return false;
  if (S.nslices <= kBSplitSlices) return true;
  return S.width > kBSplitLong && S.nslices * (int64_t)S.width * 64 >= 2 * S.slots;
}

// One row of a valued operator: entries k = 0..len-1 at stride kSlice, column
// = cb + cp[k * kSlice] (16-bit offsets) or cp[k * kSlice] (32-bit, cb = 0).
// With K > 1 the caller folds every K-th entry only: len counts those, and
// cp and vp point at the first of them.  The loads of 8 (then 4) entries are
// issued before their adds, which stay in entry order: a long row pays one
// column -> x round trip per 8 entries, and the sum keeps its bits.
template <int K = 1, typename CT, typename VT, typename XT, typename T, class Op>
__device__ __forceinline__ T sell_row(const CT* __restrict__ cp, uint32_t cb,
                                      const VT* __restrict__ vp, int len,
                                      const XT* __restrict__ x, T acc, const Op& op) {
  constexpr int S = K * kSlice;
  int k = 0;
  for (; k + 8 <= len; k += 8) {
    uint32_t c[8];
    T a[8], xv[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) c[u] = cb + cp[(k + u) * S];
#pragma unroll
    for (int u = 0; u < 8; ++u) a[u] = (T)ld(vp + (k + u) * S);
#pragma unroll
    for (int u = 0; u < 8; ++u) xv[u] = (T)x[c[u]];
#pragma unroll
    for (int u = 0; u < 8; ++u) acc = op.step(acc, a[u], xv[u]);
  }
  for (; k + 4 <= len; k += 4) {
    const uint32_t c0 = cb + cp[(k + 0) * S], c1 = cb + cp[(k + 1) * S];
    const uint32_t c2 = cb + cp[(k + 2) * S], c3 = cb + cp[(k + 3) * S];
    const T a0 = (T)ld(vp + (k + 0) * S), a1 = (T)ld(vp + (k + 1) * S);
    const T a2 = (T)ld(vp + (k + 2) * S), a3 = (T)ld(vp + (k + 3) * S);
    const T x0 = (T)x[c0], x1 = (T)x[c1], x2 = (T)x[c2], x3 = (T)x[c3];
    acc = op.step(acc, a0, x0);
    acc = op.step(acc, a1, x1);
    acc = op.step(acc, a2, x2);
    acc = op.step(acc, a3, x3);
  }
  for (; k < len; ++k) acc = op.step(acc, (T)ld(vp + k * S), (T)x[cb + cp[k * S]]);
  return acc;
}

// One row that follows a shared relative pattern: column = row + off[k]
// (the offsets come from a table of a few KB, served by the caches).  With
// K > 1, as above: every K-th entry, off and vp at the first of them.
template <int K = 1, typename VT, typename XT, typename T, class Op>
__device__ __forceinline__ T sell_row_pattern(const int32_t* __restrict__ off, uint32_t row,
                                              const VT* __restrict__ vp, int len,
                                              const XT* __restrict__ x, T acc, const Op& op) {
  constexpr int S = K * kSlice;
  int k = 0;
  for (; k + 8 <= len; k += 8) {
    uint32_t c[8];
    T a[8], xv[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) c[u] = row + off[(k + u) * K];
#pragma unroll
    for (int u = 0; u < 8; ++u) a[u] = (T)ld(vp + (k + u) * S);
#pragma unroll
    for (int u = 0; u < 8; ++u) xv[u] = (T)x[c[u]];
#pragma unroll
    for (int u = 0; u < 8; ++u) acc = op.step(acc, a[u], xv[u]);
  }
  for (; k + 4 <= len; k += 4) {
    const uint32_t c0 = row + off[(k + 0) * K], c1 = row + off[(k + 1) * K];
    const uint32_t c2 = row + off[(k + 2) * K], c3 = row + off[(k + 3) * K];
    const T a0 = (T)ld(vp + (k + 0) * S), a1 = (T)ld(vp + (k + 1) * S);
    const T a2 = (T)ld(vp + (k + 2) * S), a3 = (T)ld(vp + (k + 3) * S);
    const T x0 = (T)x[c0], x1 = (T)x[c1], x2 = (T)x[c2], x3 = (T)x[c3];
    acc = op.step(acc, a0, x0);
    acc = op.step(acc, a1, x1);
    acc = op.step(acc, a2, x2);
    acc = op.step(acc, a3, x3);
  }
  for (; k < len; ++k) acc = op.step(acc, (T)ld(vp + k * S), (T)x[row + off[k * K]]);
  return acc;
}

// One row of a slice whose 64 rows share pattern and values: offsets and values
// are wave-uniform (scalar loads), the x entry of a step is one load at a scalar
// base plus the lane's row (n < 2^29 rows, so the byte offset fits 32 bits).  The
// row length is uniform too, so the last entries' loads are all issued before
// their steps.  With K > 1, every K-th entry, off and vt at the first of them.
// No values stream from memory: the residual of the 129^3 constant-coefficient
// Q1 operator (columns sorted) takes 28 us in FP64 against 87 with its 339 MB of
// values, 17 in FP32 whatever the storage (f16 21, f32 39); what is left is the
// vectors, the row order and the x loads from the caches.
template <int K = 1, typename TV, typename XT, typename T, class Op>
__device__ __forceinline__ T sell_row_shared(const int32_t* __restrict__ off,
                                             const TV* __restrict__ vt, uint32_t row, int len,
                                             const XT* __restrict__ x, T acc, const Op& op) {
  const uint32_t at = row * (uint32_t)sizeof(XT);
  auto entry = [&](int k) {
    return (T) * reinterpret_cast<const XT*>(reinterpret_cast<const char*>(x + off[k * K]) + at);
  };
  int k = 0;
  for (; k + 8 <= len; k += 8) {
    T xv[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) xv[u] = entry(k + u);
#pragma unroll
    for (int u = 0; u < 8; ++u) acc = op.step(acc, (T)vt[(k + u) * K], xv[u]);
  }
  T xv[7];
#pragma unroll
  for (int u = 0; u < 7; ++u)
    if (k + u < len) xv[u] = entry(k + u);
#pragma unroll
  for (int u = 0; u < 7; ++u)
    if (k + u < len) acc = op.step(acc, (T)vt[(k + u) * K], xv[u]);
  return acc;
}

// type of the shared value rows of a storage type
template <typename VT>
using SharedT = typename std::conditional<std::is_same<VT, double>::value, double, float>::type;
constexpr uint32_t kSharedBit = 0x10000000u, kSharedMask = 0x0FFFFFFFu;

// valued operator (matrix); VT storage type, T arithmetic type.  A slice is one
// wavefront, so the column-encoding branch is uniform across the wave.
template <typename VT, typename XT, typename T, class Op>
__global__ __launch_bounds__(kBlock) void k_sell(int64_t n, const uint32_t* __restrict__ sptr,
                                                 const uint16_t* __restrict__ rlen,
                                                 const uint16_t* __restrict__ cidx,
                                                 const uint32_t* __restrict__ cptr,
                                                 const uint32_t* __restrict__ cbase,
                                                 const int32_t* __restrict__ ptab,
                                                 const int32_t* __restrict__ pstart,
                                                 const SharedT<VT>* __restrict__ vtab,
                                                 const VT* __restrict__ val,
                                                 const int32_t* __restrict__ perm,
                                                 const XT* __restrict__ x, Op op) {
  // Lanes past the last slot repeat slot n-1 with their own (padding) slots
  // and only skip the store, so the control flow stays uniform across the wave
  // and wave-uniform loads can use the scalar unit.  Slot t runs row perm[t]
  // (t itself without a permutation).
  const int64_t slot0 = (int64_t)xcd_block(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
  const bool active = slot0 < n;
  const int64_t slot = active ? slot0 : n - 1;
  const int64_t row = perm ? (int64_t)perm[slot] : slot;
  const int lane = threadIdx.x & (kSlice - 1);
  // the slice index is the same for the 64 lanes of a wavefront
  const int64_t s = __builtin_amdgcn_readfirstlane((int)(slot >> 6));
  const VT* vp = val + sptr[s] + lane;
  const uint32_t meta = cptr[s];
  T acc = op.init(row);
  if ((meta & 0x60000000u) == 0x60000000u) {
    // one pattern for the whole slice: wave-uniform offsets (scalar loads)
    const int pid = __builtin_amdgcn_readfirstlane((int)cbase[s]);
    const int p0 = pstart[pid];
    const int len = pstart[pid + 1] - p0;
    if (meta & kSharedBit)
      acc = sell_row_shared(ptab + p0, vtab + (meta & kSharedMask), (uint32_t)row, len, x, acc, op);
    else
      acc = sell_row_pattern(ptab + p0, (uint32_t)row, vp, len, x, acc, op);
  } else {
    const int r = rlen[slot];  // entry count, or pattern id in pattern slices
    if (meta & 0x40000000u) {
      const int p0 = pstart[r];
      acc = sell_row_pattern(ptab + p0, (uint32_t)row, vp, pstart[r + 1] - p0, x, acc, op);
    } else if (meta & 0x80000000u) {
      acc = sell_row((const uint32_t*)(cidx + (meta & 0x1FFFFFFFu)) + lane, 0u, vp, r, x, acc, op);
    } else {
      acc = sell_row(cidx + meta + lane, cbase[s], vp, r, x, acc, op);
    }
  }
  if (active) op.finish(row, acc);
}

// The same sweep for reduced-precision (non-exact) ops on levels with few
// slices, where one thread per row leaves the chip mostly idle and each row
// is a long chain of dependent loads (Q2 rows hold up to 125 entries).  A
// workgroup of K wavefronts takes one slice: wavefront w folds entries
// w, w + K, w + 2K, ... of each of the slice's 64 rows (every load still
// covers 64 contiguous slots), and wavefront 0 adds the K partial sums, in
// order, to the row's start value.  Each partial chain starts from zero,
// which is right for ops whose step is acc + a x or acc - a x (SpmvOp,
// ResidualOp, JacobiOp).  That reorders the row sum, so exact ops are
// rejected at compile time.  Every thread reaches the barrier: lanes past
// the last row repeat row n-1, as in k_sell, and only skip the store.
template <typename VT, typename XT, typename T, class Op, int K>
__global__ __launch_bounds__(kSlice * K) void k_sell_split(
    int64_t n, const uint32_t* __restrict__ sptr, const uint16_t* __restrict__ rlen,
    const uint16_t* __restrict__ cidx, const uint32_t* __restrict__ cptr,
    const uint32_t* __restrict__ cbase, const int32_t* __restrict__ ptab,
    const int32_t* __restrict__ pstart, const SharedT<VT>* __restrict__ vtab,
    const VT* __restrict__ val,
    const int32_t* __restrict__ perm, const XT* __restrict__ x, Op op) {
  static_assert(!Op::kExact, "split sweeps reorder the row sums");
  __shared__ T part[K][kSlice];
  const int64_t s = xcd_block(blockIdx.x, gridDim.x);  // one slice per workgroup
  const int lane = threadIdx.x & (kSlice - 1);
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kSlice));
  const int64_t slot0 = s * kSlice + lane;
  const bool active = slot0 < n;
  const int64_t slot = active ? slot0 : n - 1;
  const int64_t row = perm ? (int64_t)perm[slot] : slot;
  const VT* vp = val + sptr[s] + lane + w * kSlice;
  const uint32_t meta = cptr[s];
  // entries w, w + K, ... below len
  auto mine = [w](int len) { return len > w ? (len - w + K - 1) / K : 0; };
  T acc = (T)0;
  if ((meta & 0x60000000u) == 0x60000000u) {
    const int pid = __builtin_amdgcn_readfirstlane((int)cbase[s]);
    const int p0 = pstart[pid];
    const int len = mine(pstart[pid + 1] - p0);
    if (meta & kSharedBit)
      acc = sell_row_shared<K>(ptab + p0 + w, vtab + (meta & kSharedMask) + w, (uint32_t)row, len,
                               x, acc, op);
    else
      acc = sell_row_pattern<K>(ptab + p0 + w, (uint32_t)row, vp, len, x, acc, op);
  } else {
    const int r = rlen[slot];
    if (meta & 0x40000000u) {
      const int p0 = pstart[r];
      acc = sell_row_pattern<K>(ptab + p0 + w, (uint32_t)row, vp, mine(pstart[r + 1] - p0), x,
                                acc, op);
    } else if (meta & 0x80000000u) {
      acc = sell_row<K>((const uint32_t*)(cidx + (meta & 0x1FFFFFFFu)) + lane + w * kSlice, 0u,
                        vp, mine(r), x, acc, op);
    } else {
      acc = sell_row<K>(cidx + meta + lane + w * kSlice, cbase[s], vp, mine(r), x, acc, op);
    }
  }
  part[w][lane] = acc;
  __syncthreads();
  if (w == 0) {
    T sum = op.init(row);
#pragma unroll
    for (int i = 0; i < K; ++i) sum += part[i][lane];
    if (active) op.finish(row, sum);
  }
}

// k_sell for exact ops on long rows, whose chains of loads and scattered gathers
// (caller's entry order) bound one wavefront per slice: a workgroup of K wavefronts
// per slice forms the rounded products of K * E entries of the 64 rows at a time,
// side by side, into LDS, and wavefront 0 folds them into the rows in entry
// order -- the additions of k_sell in the same order, bit for bit.  Entry k of a
// round goes to wavefront k % K.  Entries past the slice's width repeat its last
// one (their values and columns exist), and every product past a row's end is
// replaced by the fold's neutral element.  The loads run ahead of the fold: while
// a round is folded the next one's values and x entries and the columns after
// that are in flight.  Two buffers, one barrier per round.
template <typename VT, typename XT, typename T, class Op, int K>
__global__ __launch_bounds__(kSlice * K) void k_sell_fold(
    int64_t n, const uint32_t* __restrict__ sptr, const uint16_t* __restrict__ rlen,
    const uint16_t* __restrict__ cidx, const uint32_t* __restrict__ cptr,
    const uint32_t* __restrict__ cbase, const int32_t* __restrict__ ptab,
    const int32_t* __restrict__ pstart, const SharedT<VT>* __restrict__ vtab,
    const VT* __restrict__ val,
    const int32_t* __restrict__ perm, const XT* __restrict__ x, Op op) {
  constexpr int E = 8, C = K * E;
  __shared__ T part[2][C][kSlice];
  const int64_t s = xcd_block(blockIdx.x, gridDim.x);  // one slice per workgroup
  const int lane = threadIdx.x & (kSlice - 1);
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kSlice));
  const int64_t slot0 = s * kSlice + lane;
  const bool active = slot0 < n;
  const int64_t slot = active ? slot0 : n - 1;
  const int64_t row = perm ? (int64_t)perm[slot] : slot;
  const uint32_t v0 = sptr[s];
  const int width = (int)((sptr[s + 1] - v0) / kSlice);
  const VT* vp = val + v0 + lane;
  const uint32_t meta = cptr[s];
  const uint32_t cb = cbase[s];
  const bool patterned = (meta & 0x40000000u) != 0, wide = (meta & 0x80000000u) != 0;
  int len = 0;
  const int32_t* off = ptab;
  if (patterned) {
    const int pid = (meta & 0x20000000u) ? __builtin_amdgcn_readfirstlane((int)cb) : (int)rlen[slot];
    const int p0 = pstart[pid];
    off = ptab + p0;
    len = pstart[pid + 1] - p0;
  } else {
    len = rlen[slot];
  }
  const uint16_t* c16 = cidx + (meta & 0x1FFFFFFFu) + lane;
  const uint32_t* c32 = (const uint32_t*)(cidx + (meta & 0x1FFFFFFFu)) + lane;
  uint32_t c[E];
  T a[E], xv[E];
  auto columns = [&](int c0) {
    if (patterned) {
#pragma unroll
      for (int u = 0; u < E; ++u) {
        const int k = c0 + u * K + w;
        c[u] = (uint32_t)row + (k < len ? off[k] : 0);
      }
    } else if (wide) {
#pragma unroll
      for (int u = 0; u < E; ++u) c[u] = c32[(int64_t)min(c0 + u * K + w, width - 1) * kSlice];
    } else {
#pragma unroll
      for (int u = 0; u < E; ++u)
        c[u] = cb + c16[(int64_t)min(c0 + u * K + w, width - 1) * kSlice];
    }
  };
  const bool shared = (meta & 0x70000000u) == 0x70000000u;
  const SharedT<VT>* vt = vtab + (shared ? meta & kSharedMask : 0u);
  auto entries = [&](int c0) {
    if (shared) {  // (as many entries as the slice is wide, the same for every row)
#pragma unroll
      for (int u = 0; u < E; ++u) a[u] = (T)vt[min(c0 + u * K + w, width - 1)];
    } else {
#pragma unroll
      for (int u = 0; u < E; ++u)
        a[u] = (T)ld(vp + (int64_t)min(c0 + u * K + w, width - 1) * kSlice);
    }
#pragma unroll
    for (int u = 0; u < E; ++u) xv[u] = (T)x[c[u]];
  };
  T acc = (T)0;
  if (w == 0) acc = op.init(row);
  if (width > 0) {
    columns(0);
    entries(0);
    if (C < width) columns(C);
  }
  for (int c0 = 0, buf = 0; c0 < width; c0 += C, buf ^= 1) {
#pragma unroll
    for (int u = 0; u < E; ++u)
      part[buf][u * K + w][lane] = c0 + u * K + w < len ? mul_rn(a[u], xv[u]) : Op::neutral();
    __syncthreads();
    if (c0 + C < width) entries(c0 + C);
    if (c0 + 2 * C < width) columns(c0 + 2 * C);
    __builtin_amdgcn_sched_barrier(0);
    if (w == 0) {
#pragma unroll
      for (int u0 = 0; u0 < C; u0 += 16) {
        if (c0 + u0 < width) {
          T q[16];
#pragma unroll
          for (int u = 0; u < 16; ++u) q[u] = part[buf][u0 + u][lane];
#pragma unroll
          for (int u = 0; u < 16; ++u) acc = op.fold(acc, q[u]);
        }
      }
    }
  }
  if (w == 0 && active) op.finish(row, acc);
}

// Wavefronts per slice of an exact sweep (0: k_sell).  The fold pays where the
// chains of long rows bound the sweep, FP64 residuals, k_sell / 4 / 8 wavefronts:
//  * Few slices: 8 wavefronts take 64 entries per round, their 64 KB of LDS leave a
//    CU two workgroups; 4 take 32 and leave five.  The longer the rows, the more
//    rounds 8 save and the more slices that pays for.  Q2 (125 to 285 entries at
//    most), 12 slices 8.3 / 6.5 / 5.4 us, 562 slices 13.1 / 10.7 / 10.0, 1231 slices
//    39 / 25.4 / 24.0; rows of 48, 125 slices 5.4 / 4.2 / 4.0, 469 slices 5.7 / 4.7 /
//    5.3; of 96, 469 slices 9.2 / 6.2 / 6.8; of 51 (Q1 with hanging nodes, mean 18),
//    342 slices 6.4 / 5.1 / 5.6.
//  * Many slices: only where rows of more than 64 entries are well above the mean,
//    so that few wavefronts of k_sell would hold most of the entries.  Q2, 275 K
//    rows 60 / 44 / 54, 352 K 109 / 60 / 75.  Rows of 27 and up to 51 entries lose:
//    532 K adaptive Q1 rows 25 / 36 / 67; rows of 27 and 48, 60 K 6.2 / 6.9 / 8.7.  So
//    do equal rows: 96 entries each, 120 K 22.7 / 24.6 / 30.1.
//  * Single-pattern slices take their columns from scalar registers, k_sell's loads
//    then wait for nothing: rows of 27 and 96, 120 K rows 14.3 / 17.3 / 23.0 against
//    19.2 / 17.6 / 23.0 with columns in memory.  Where they hold most of the entries,
//    the fold is for few slices only.
//  * Ascending columns gather from fewer lines than a caller's order, and enough
//    slices hide what is left: Q2 with hanging nodes, 352 K rows 86 / 56 against
//    109 / 61 in the caller's order, but 1.96 M rows (30.7 K slices) 303 / 331
//    against 400 / 360, and A z with an FP32 z 294 / 349.
constexpr int kFoldRow = 32, kFoldLong = 64;
constexpr int64_t kFoldSlices4 = 512, kFoldSlicesAscending = 16384;
inline int sell_fold_waves(const Sell& S) {
  if (S.maxlen <= kFoldRow) return 0;
  if (S.nslices <= 5 * (int64_t)S.maxlen) return 8;
  if (2 * S.single > S.slots) return 0;
  if (S.nslices <= kFoldSlices4) return 4;
  if (S.ascending && S.nslices > kFoldSlicesAscending) return 0;
  return S.maxlen > kFoldLong && 2 * S.nslices * S.maxlen * kSlice >= 3 * S.slots ? 4 : 0;
}

// Split factor of a reduced-precision sweep: double K while the level runs
// fewer than 8192 wavefronts (32 per CU) and every wavefront still gets at
// least 8 of the longest row's entries, up to 16 wavefronts per slice.
inline int sell_split(const Sell& S) {
  int K = 1;
  while (K < 16 && S.nslices * K < 8192 && S.maxlen >= 16 * K) K *= 2;
  return K;
}

// packed-weight operator (grid transfer): w = 2^-code from the column's top bits
template <typename T, class Op>
__global__ __launch_bounds__(kBlock) void k_sell_w(int64_t n, const uint32_t* __restrict__ sptr,
                                                   const uint16_t* __restrict__ rlen,
                                                   const uint32_t* __restrict__ col,
                                                   const T* __restrict__ x, Op op) {
  const int64_t row = (int64_t)xcd_block(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
  if (row >= n) return;
  const int lane = threadIdx.x & (kSlice - 1);
  const uint32_t* cp = col + sptr[row >> 6] + lane;
  const int len = rlen[row];
  T acc = op.init(row);
  int k = 0;
  for (; k + 4 <= len; k += 4) {
    const uint32_t e0 = cp[(k + 0) * kSlice], e1 = cp[(k + 1) * kSlice];
    const uint32_t e2 = cp[(k + 2) * kSlice], e3 = cp[(k + 3) * kSlice];
    const T x0 = x[e0 & kIdxMask], x1 = x[e1 & kIdxMask], x2 = x[e2 & kIdxMask],
            x3 = x[e3 & kIdxMask];
    acc = op.step(acc, code_weight<T>(e0 >> 29), x0);
    acc = op.step(acc, code_weight<T>(e1 >> 29), x1);
    acc = op.step(acc, code_weight<T>(e2 >> 29), x2);
    acc = op.step(acc, code_weight<T>(e3 >> 29), x3);
  }
  for (; k < len; ++k) {
    const uint32_t e = cp[k * kSlice];
    acc = op.step(acc, code_weight<T>(e >> 29), x[e & kIdxMask]);
  }
  op.finish(row, acc);
}

// The grid transfers of an FP32 V-cycle on levels of few slices, split as
// k_sell_split splits the sweeps: wavefront w of a slice's K folds entries
// w, w + K, ... of each row from zero, and wavefront 0 adds the K partial sums,
// in order, to op.init(row).  Every transfer op steps acc + w x, so only the
// order of the row sum changes; the FP64 transfers keep one thread per row and
// their bits.
template <typename T, class Op, int K>
__global__ __launch_bounds__(kSlice * K) void k_sell_w_split(int64_t n,
                                                             const uint32_t* __restrict__ sptr,
                                                             const uint16_t* __restrict__ rlen,
                                                             const uint32_t* __restrict__ col,
                                                             const T* __restrict__ x, Op op) {
  __shared__ T part[K][kSlice];
  const int64_t s = xcd_block(blockIdx.x, gridDim.x);  // one slice per workgroup
  const int lane = threadIdx.x & (kSlice - 1);
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kSlice));
  const int64_t row0 = s * kSlice + lane;
  const bool active = row0 < n;
  const int64_t row = active ? row0 : n - 1;
  const uint32_t* cp = col + sptr[s] + lane + w * kSlice;
  const int len = rlen[row];
  const int mine = len > w ? (len - w + K - 1) / K : 0;
  constexpr int S = K * kSlice;
  T acc = (T)0;
  int k = 0;
  for (; k + 4 <= mine; k += 4) {
    const uint32_t e0 = cp[(k + 0) * S], e1 = cp[(k + 1) * S];
    const uint32_t e2 = cp[(k + 2) * S], e3 = cp[(k + 3) * S];
    const T x0 = x[e0 & kIdxMask], x1 = x[e1 & kIdxMask], x2 = x[e2 & kIdxMask],
            x3 = x[e3 & kIdxMask];
    acc = op.step(acc, code_weight<T>(e0 >> 29), x0);
    acc = op.step(acc, code_weight<T>(e1 >> 29), x1);
    acc = op.step(acc, code_weight<T>(e2 >> 29), x2);
    acc = op.step(acc, code_weight<T>(e3 >> 29), x3);
  }
  for (; k < mine; ++k) {
    const uint32_t e = cp[k * S];
    acc = op.step(acc, code_weight<T>(e >> 29), x[e & kIdxMask]);
  }
  part[w][lane] = acc;
  __syncthreads();
  if (w == 0) {
    T sum = op.init(row);
#pragma unroll
    for (int i = 0; i < K; ++i) sum += part[i][lane];
    if (active) op.finish(row, sum);
  }
}

// Split factor of an FP32 transfer: double K while the doubled level still
// runs at most 8192 wavefronts and every wavefront still gets at least 4 of
// the longest row's entries, up to 16.  (Levels of more than 4096 slices stay
// unsplit: at 64^3 a split of 2 measured slower than one thread per row.)
inline int sell_w_split(const Sell& S) {
  int K = 1;
  while (K < 16 && S.nslices * 2 * K <= 8192 && S.maxlen >= 4 * K) K *= 2;
  return K;
}

template <typename T, class Op, int K>
inline int sell_w_split_launch(gh_ctx* ctx, const Sell& S, const T* x, Op op) {
  hipLaunchKernelGGL((k_sell_w_split<T, Op, K>), dim3((unsigned)S.nslices), dim3(kSlice * K), 0,
                     ctx->stream, S.n, S.sptr, S.rlen, S.col, x, op);
  GH_HIP(hipGetLastError());
  return GH_OK;
}

template <typename VT, typename XT, typename T, class Op, int K>
inline int sell_fold_launch(gh_ctx* ctx, const Sell& S, const XT* x, Op op) {
  hipLaunchKernelGGL((k_sell_fold<VT, XT, T, Op, K>), dim3((unsigned)S.nslices), dim3(kSlice * K),
                     0, ctx->stream, S.n, S.sptr, S.rlen, S.cidx, S.cptr, S.cbase, S.ptab,
                     S.pstart, (const SharedT<VT>*)S.vtab, (const VT*)S.val, S.perm, x, op);
  GH_HIP(hipGetLastError());
  return GH_OK;
}

template <typename VT, typename XT, typename T, class Op, int K>
inline int sell_split_launch(gh_ctx* ctx, const Sell& S, const XT* x, Op op) {
  hipLaunchKernelGGL((k_sell_split<VT, XT, T, Op, K>), dim3((unsigned)S.nslices),
                     dim3(kSlice * K), 0, ctx->stream, S.n, S.sptr, S.rlen, S.cidx, S.cptr,
                     S.cbase, S.ptab, S.pstart, (const SharedT<VT>*)S.vtab, (const VT*)S.val, S.perm, x, op);
  GH_HIP(hipGetLastError());
  return GH_OK;
}

template <typename VT, typename XT, typename T, class Op>
inline int sell_launch(gh_ctx* ctx, const Sell& S, const XT* x, Op op) {
  if (S.n == 0) return GH_OK;
  if constexpr (!Op::kExact) {
    switch (sell_split(S)) {
      case 2: return sell_split_launch<VT, XT, T, Op, 2>(ctx, S, x, op);
      case 4: return sell_split_launch<VT, XT, T, Op, 4>(ctx, S, x, op);
      case 8: return sell_split_launch<VT, XT, T, Op, 8>(ctx, S, x, op);
      case 16: return sell_split_launch<VT, XT, T, Op, 16>(ctx, S, x, op);
      default: break;
    }
  } else {
    switch (sell_fold_waves(S)) {
      case 4: return sell_fold_launch<VT, XT, T, Op, 4>(ctx, S, x, op);
      case 8: return sell_fold_launch<VT, XT, T, Op, 8>(ctx, S, x, op);
      default: break;
    }
  }
  hipLaunchKernelGGL((k_sell<VT, XT, T, Op>), dim3(grid_for(S.n)), dim3(kBlock), 0, ctx->stream,
                     S.n, S.sptr, S.rlen, S.cidx, S.cptr, S.cbase, S.ptab, S.pstart,
                     (const SharedT<VT>*)S.vtab, (const VT*)S.val, S.perm, x, op);
  GH_HIP(hipGetLastError());
  return GH_OK;
}

template <typename XT, typename T, class Op>
inline int sell_dispatch(gh_ctx* ctx, const Sell& S, const XT* x, Op op) {
  if (S.prec == GH_F64) return sell_launch<double, XT, T, Op>(ctx, S, x, op);
  if (S.prec == GH_F32) return sell_launch<float, XT, T, Op>(ctx, S, x, op);
  return sell_launch<__half, XT, T, Op>(ctx, S, x, op);
}

template <typename T, class Op>
inline int sell_w_launch(gh_ctx* ctx, const Sell& S, const T* x, Op op) {
  if (S.n == 0) return GH_OK;
  if constexpr (std::is_same<T, float>::value) {
    switch (sell_w_split(S)) {
      case 2: return sell_w_split_launch<T, Op, 2>(ctx, S, x, op);
      case 4: return sell_w_split_launch<T, Op, 4>(ctx, S, x, op);
      case 8: return sell_w_split_launch<T, Op, 8>(ctx, S, x, op);
      case 16: return sell_w_split_launch<T, Op, 16>(ctx, S, x, op);
      default: break;
    }
  }
  hipLaunchKernelGGL((k_sell_w<T, Op>), dim3(grid_for(S.n)), dim3(kBlock), 0, ctx->stream, S.n,
                     S.sptr, S.rlen, S.col, x, op);
  GH_HIP(hipGetLastError());
  return GH_OK;
}

}  // namespace gh
