// Vanka patch smoother (src/LinAlg/vankasmoother.cc): the patch matrices of a
// node-block matrix, LU with partial pivoting on the device, and the solve
//   x <- (1/count_i) sum_p R_p^T A_p^-1 R_p x.
// Factoring: one workgroup of 1024 threads per patch, the m x m patch matrix
// (m <= 128) in the threads' registers, the LU's operations uncontracted so
// that the factors equal the oracle's; the recorded row exchanges are composed on the host into
// one gather per factor row.  Patches with equal matrices are found first and
// factored once.  Solving: column-oriented triangular solves of the local
// vector, gathered in pivoted order, by one of two kernels: grouped (the
// factors of one class in LDS, 16 lanes per patch, k_vanka_group) or streamed
// (one wavefront per patch reading its own factors, k_vanka_solve).  Averaging:
// one thread per unknown, the patches containing its node added in ascending
// order (the reference adds with OpenMP atomics, in no fixed order).
#include <algorithm>
#include <cmath>
#include <vector>

#include "gh_kernels.h"

using namespace gh;

namespace {

constexpr int kVankaMaxM = 128;       // local unknowns per patch
constexpr int kVankaMaxNodes = 128;   // nodes per patch

// Factoring one patch: 1024 threads, lane tr = t % 64 of wavefront tc = t / 64
// keeps the entries (tr + 64 i, tc + 16 j), i < 2, j < 8, of the m x m patch
// matrix (m <= 128) in registers, so the 64 owners of a column form one
// wavefront and its pivot search is a wavefront reduction.  Row exchanges are
// not carried out: every thread keeps the position of each of its rows in the
// exchanged order, and the factors are written in that order at the end.
// LDS holds only the patch's CSR positions and, per column, the multipliers
// and the pivot (double-buffered), a few KB, so two patches share a CU.
constexpr int kFactorThreads = 1024;
constexpr int kFactorLanes = 64;                          // rows tr + 64 i
constexpr int kFactorWaves = kFactorThreads / kFactorLanes;  // columns tc + 16 j
constexpr int kRowsPer = kVankaMaxM / kFactorLanes;       // 2
constexpr int kColsPer = kVankaMaxM / kFactorWaves;       // 8

struct FactorShared {
  double l[2][kVankaMaxM];  // the multipliers of the column, by row
  int32_t pr[2], rp[2];     // the pivot's position before the exchange, and its row
  double d[2];              // the pivot
};

// Columns 16 KB .. 16 KB + 15 (KB a constant, so that the column's registers
// are known): per column k, one barrier.
//   A: the wavefront owning column k (already updated by itself) finds the
//      pivot by a maximum of |a_ik| and a minimum of position * 256 + row,
//      forms the multipliers, puts them and the pivot into LDS, records
//      piv[k];
//   B: every thread exchanges the positions k and piv[k] among its rows and
//      updates its entries below and right of (k, k): the pivot row's entries
//      in a wavefront's columns are held by one of its own lanes (rp % 64),
//      which broadcasts them.
// The buffers alternate between columns, so the owner of column k + 1 may
// start before the others have finished column k.
template <int KB>
__device__ __forceinline__ void factor_columns(int m, int tr, int tc,
                                               double (&a)[kRowsPer][kColsPer],
                                               int (&pos)[kRowsPer], FactorShared& S,
                                               int32_t* __restrict__ pv) {
  for (int kk = 0; kk < kFactorWaves; ++kk) {
    const int k = KB * kFactorWaves + kk;
    if (k >= m) return;
    const int buf = k & 1;
    if (tc == kk) {
      double best = -1.0;  // fmax passes NaN over
#pragma unroll
      for (int i = 0; i < kRowsPer; ++i)
        if (pos[i] >= k) best = fmax(best, fabs(a[i][KB]));
      best = wave_max_nonneg(best);
      // the smallest position holding the maximum (a NaN a_kk keeps row k, as
      // the oracle's strict comparisons do); a key always exists, since a
      // non-NaN a_kk makes best >= |a_kk| attained
      int key = INT_MAX;
#pragma unroll
      for (int i = 0; i < kRowsPer; ++i) {
        const double v = a[i][KB];
        const bool cand = pos[i] > k ? fabs(v) == best
                                     : pos[i] == k && (fabs(v) == best || v != v);
        if (cand) key = min(key, pos[i] * 256 + tr + kFactorLanes * i);
      }
      key = wave_min(key);
      const int pr = key >> 8, rp = key & 255;
      const double d = lane_read(rp < kFactorLanes ? a[0][KB] : a[1][KB], rp % kFactorLanes);
      if (d != 0.0) {
#pragma unroll
        for (int i = 0; i < kRowsPer; ++i) {
          const int r = tr + kFactorLanes * i;
          if (pos[i] >= k && r != rp) {
            const double l = a[i][KB] / d;
            a[i][KB] = l;
            S.l[buf][r] = l;
          }
        }
      }
      if (tr == 0) {
        S.pr[buf] = pr;
        S.rp[buf] = rp;
        S.d[buf] = d;
        pv[k] = pr;
      }
    }
    __syncthreads();
    const int pr = __builtin_amdgcn_readfirstlane(S.pr[buf]);
    const int rp = __builtin_amdgcn_readfirstlane(S.rp[buf]);
    const double d = S.d[buf];
#pragma unroll
    for (int i = 0; i < kRowsPer; ++i) {
      const int r = tr + kFactorLanes * i;
      pos[i] = (r == rp) ? k : (pos[i] == k ? pr : pos[i]);
    }
    if (d != 0.0) {
      double l[kRowsPer];
#pragma unroll
      for (int i = 0; i < kRowsPer; ++i) l[i] = pos[i] > k ? S.l[buf][tr + kFactorLanes * i] : 0.0;
#pragma unroll
      for (int j = KB; j < kColsPer; ++j) {
        // column tc + 16 j > k: every j > KB, and j = KB right of the pivot
        if (!((j > KB || tc > kk) && tc + kFactorWaves * j < m)) continue;
        // the pivot row's entry in this column, from the lane holding it
        const double u = lane_read(rp < kFactorLanes ? a[0][j] : a[1][j], rp % kFactorLanes);
#pragma unroll
        for (int i = 0; i < kRowsPer; ++i)
          if (pos[i] > k) a[i][j] = add_rn(a[i][j], -mul_rn(l[i], u));
      }
    }
  }
}

// A patch's nodes and their places, open addressing (at most half full).
struct PatchMap {
  static constexpr int kSize = 2 * kVankaMaxNodes;
  int32_t node[kSize], place[kSize];
  static __device__ __forceinline__ int hash(int32_t v) {
    return (int)(((uint32_t)v * 0x9E3779B1u) >> 24);
  }
};
static_assert(PatchMap::kSize == 256, "hash: 8 bits");

// copy_entries_sparseblockmatrix: tab[r * psize + u] = CSR position of the block
// (patch node r, patch node u), -1 where the matrix has none.  All NT threads of
// the workgroup; NT / psize of them walk each row's entries and look the columns
// up.  Ends in a barrier.
template <int NT>
__device__ __forceinline__ void patch_positions(int psize, const int32_t* __restrict__ nodes,
                                                const int32_t* __restrict__ rowptr,
                                                const int32_t* __restrict__ col, int32_t* tab,
                                                PatchMap& map) {
  constexpr int last = PatchMap::kSize - 1;
  const int t = threadIdx.x;
  for (int e = t; e < psize * psize; e += NT) tab[e] = -1;
  for (int e = t; e <= last; e += NT) map.node[e] = -1;
  __syncthreads();
  for (int r = t; r < psize; r += NT) {  // distinct nodes: each takes a free slot
    int h = PatchMap::hash(nodes[r]);
    while (atomicCAS(&map.node[h], -1, nodes[r]) != -1) h = (h + 1) & last;
    map.place[h] = r;
  }
  __syncthreads();
  const int per = NT / psize;
  const int r = t / per, u0 = t - r * per;
  if (r < psize) {
    const int32_t row = nodes[r];
    for (int32_t q = rowptr[row] + u0; q < rowptr[row + 1]; q += per) {
      const int32_t c0 = col[q];
      int h = PatchMap::hash(c0);
      while (map.node[h] != c0 && map.node[h] != -1) h = (h + 1) & last;
      if (map.node[h] == c0) tab[r * psize + map.place[h]] = q;
    }
  }
  __syncthreads();
}

// the 64-bit finaliser of SplitMix64
__device__ __forceinline__ uint64_t mix64(uint64_t z) {
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

constexpr int kHashThreads = 1024;  // as many walk a row: 64 patches of 108, creation 0.34 ms with 256

// Two 64-bit sums over the patch matrix's entries, each entry's bits mixed with
// its place: equal matrices have equal sums, and the patches with equal sums are
// compared entry by entry afterwards (k_vanka_same).
__global__ __launch_bounds__(kHashThreads) void k_vanka_hash(
    int psize, int B, const int32_t* __restrict__ nodes, const int32_t* __restrict__ rowptr,
    const int32_t* __restrict__ col, const double* __restrict__ val, uint64_t* __restrict__ out) {
  extern __shared__ int32_t tab[];
  __shared__ PatchMap map;
  __shared__ uint64_t part[2][kHashThreads / 64];
  const int64_t p = blockIdx.x;
  const int BB = B * B, t = threadIdx.x;
  patch_positions<kHashThreads>(psize, nodes + p * psize, rowptr, col, tab, map);
  uint64_t h0 = 0, h1 = 0;
  for (int e = t; e < psize * psize * BB; e += kHashThreads) {
    const int32_t q = tab[e / BB];
    const double x = q >= 0 ? val[(int64_t)q * BB + e % BB] : 0.0;
    const uint64_t b = __builtin_bit_cast(uint64_t, x);
    h0 += mix64(b + (uint64_t)(e + 1) * 0x9E3779B97F4A7C15ull);
    h1 += mix64((b ^ 0xD1B54A32D192ED03ull) + (uint64_t)(e + 1) * 0xABC98388FB8FAC03ull);
  }
  for (int off = 32; off > 0; off >>= 1) {
    h0 += (uint64_t)__shfl_down((unsigned long long)h0, off, 64);
    h1 += (uint64_t)__shfl_down((unsigned long long)h1, off, 64);
  }
  if ((t & 63) == 0) {
    part[0][t >> 6] = h0;
    part[1][t >> 6] = h1;
  }
  __syncthreads();
  if (t < 2) {
    uint64_t s = 0;
    for (int w = 0; w < kHashThreads / 64; ++w) s += part[t][w];
    out[2 * p + t] = s;
  }
}

// flag[p]: whether patch p's matrix differs from patch rep[p]'s in any bit
__global__ __launch_bounds__(kHashThreads) void k_vanka_same(
    int psize, int B, const int32_t* __restrict__ nodes, const int32_t* __restrict__ rowptr,
    const int32_t* __restrict__ col, const double* __restrict__ val,
    const int32_t* __restrict__ rep, int32_t* __restrict__ flag) {
  extern __shared__ int32_t tab[];  // 2 * psize * psize
  __shared__ PatchMap map;
  const int64_t p = blockIdx.x, r = rep[p];
  if (r == p) {  // the whole workgroup
    if (threadIdx.x == 0) flag[p] = 0;
    return;
  }
  const int BB = B * B, PP = psize * psize;
  patch_positions<kHashThreads>(psize, nodes + p * psize, rowptr, col, tab, map);
  patch_positions<kHashThreads>(psize, nodes + r * psize, rowptr, col, tab + PP, map);
  int differs = 0;
  for (int e = threadIdx.x; e < PP * BB; e += kHashThreads) {
    const int32_t q = tab[e / BB], s = tab[PP + e / BB];
    const double x = q >= 0 ? val[(int64_t)q * BB + e % BB] : 0.0;
    const double y = s >= 0 ? val[(int64_t)s * BB + e % BB] : 0.0;
    differs |= __builtin_bit_cast(uint64_t, x) != __builtin_bit_cast(uint64_t, y);
  }
  differs = __syncthreads_or(differs);
  if (threadIdx.x == 0) flag[p] = differs;
}

// LU with partial pivoting of every class's patch matrix, the oracle's operations in
// the oracle's order per entry: pivot = the first row (in the exchanged order)
// of largest |a_ik|, i >= k; no elimination when the pivot is 0;
// l_i = a_ik / d and a_ij -= l_i a_kj, product and difference rounded
// separately.  (8 waves per SIMD: two patches per CU, at most 64 VGPRs.)
__global__ __launch_bounds__(kFactorThreads, 8) void k_vanka_factor(
    int psize, int B, const int32_t* __restrict__ reps, const int32_t* __restrict__ nodes,
    const int32_t* __restrict__ rowptr, const int32_t* __restrict__ col,
    const double* __restrict__ val, int ld, double* __restrict__ lu64,
    float* __restrict__ lu32, int32_t* __restrict__ piv) {
  extern __shared__ int32_t tab[];  // psize * psize CSR positions of the node blocks, -1: none
  __shared__ PatchMap map;
  __shared__ FactorShared S;
  const int64_t p = blockIdx.x;
  const int m = psize * B;
  const int t = threadIdx.x, tr = t % kFactorLanes, tc = t / kFactorLanes;
  patch_positions<kFactorThreads>(psize, nodes + (int64_t)reps[p] * psize, rowptr, col, tab, map);
  double a[kRowsPer][kColsPer];
  int pos[kRowsPer];  // position of row tr + 64 i in the exchanged order; -1: no row
#pragma unroll
  for (int i = 0; i < kRowsPer; ++i) {
    const int r = tr + kFactorLanes * i;
    pos[i] = r < m ? r : -1;
#pragma unroll
    for (int j = 0; j < kColsPer; ++j) {
      const int c = tc + kFactorWaves * j;
      double x = 0.0;
      if (r < m && c < m) {
        const int32_t q = tab[(r / B) * psize + c / B];
        if (q >= 0) x = val[((int64_t)q * B + r % B) * B + c % B];
      }
      a[i][j] = x;
    }
  }
  int32_t* pv = piv + p * m;
  factor_columns<0>(m, tr, tc, a, pos, S, pv);
  factor_columns<1>(m, tr, tc, a, pos, S, pv);
  factor_columns<2>(m, tr, tc, a, pos, S, pv);
  factor_columns<3>(m, tr, tc, a, pos, S, pv);
  factor_columns<4>(m, tr, tc, a, pos, S, pv);
  factor_columns<5>(m, tr, tc, a, pos, S, pv);
  factor_columns<6>(m, tr, tc, a, pos, S, pv);
  factor_columns<7>(m, tr, tc, a, pos, S, pv);
  // column-major factors (coalesced column reads in the solve), rows in the
  // exchanged order
  const int64_t base = p * (int64_t)ld * m;
  for (int e = t; e < (ld - m) * m; e += kFactorThreads) {  // zeros below row m
    const int64_t z = base + (int64_t)(e / (ld - m)) * ld + m + e % (ld - m);
    if (lu64) lu64[z] = 0.0;
    else lu32[z] = 0.0f;
  }
#pragma unroll
  for (int i = 0; i < kRowsPer; ++i) {
    if (pos[i] < 0) continue;
#pragma unroll
    for (int j = 0; j < kColsPer; ++j) {
      const int c = tc + kFactorWaves * j;
      if (c >= m) continue;
      const int64_t e = base + (int64_t)c * ld + pos[i];
      if (lu64) lu64[e] = a[i][j];
      else lu32[e] = (float)a[i][j];
    }
  }
}

template <typename T>
__device__ __forceinline__ T bcast(T v, int lane) {
  if constexpr (sizeof(T) == 8) {
    const int64_t b = __builtin_bit_cast(int64_t, v);
    const int lo = __builtin_amdgcn_readlane((int)(b & 0xFFFFFFFF), lane);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
    return __builtin_bit_cast(T, ((int64_t)hi << 32) | (uint32_t)lo);
  } else {
    return __builtin_bit_cast(T, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
  }
}

// reciprocals of the diagonal of U for the solves' divisions; 0 where
// a plain division is needed (zero or extreme diagonals)
template <typename T>
__global__ __launch_bounds__(kBlock) void k_vanka_rdiag(int64_t nclasses, int m, int ld,
                                                        const T* __restrict__ lu,
                                                        double* __restrict__ rdiag) {
  const int64_t t = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (t >= nclasses * m) return;
  const int64_t c = t / m;
  const int k = (int)(t - c * m);
  const double d = (double)lu[(c * m + k) * ld + k];
  const double a = fabs(d);
  rdiag[t] = (a >= 0x1p-400 && a <= 0x1p400) ? 1.0 / d : 0.0;
}

// x / d rounded to nearest, r = 1 / d rounded to nearest.  FP64: two residual
// corrections of x r (P. Markstein, IBM J. Res. Dev. 34 (1990): with r correctly
// rounded and q within an ulp of x / d, fma(x - q d, r, q) is x / d correctly
// rounded), 5 dependent operations; up to the sign of a zero the quotients are
// the division's, so the solves keep the oracle's values.  FP32: the product
// with the FP64 reciprocal.
__device__ __forceinline__ double divide_by(double x, double d, double r) {
  const double q0 = x * r;
  const double q1 = __builtin_fma(__builtin_fma(-q0, d, x), r, q0);
  return __builtin_fma(__builtin_fma(-q1, d, x), r, q1);
}
__device__ __forceinline__ float divide_by(float x, double, double r) {
  return (float)((double)x * r);
}
// whether the quotient q of divide_by, by a diagonal within 2^-400 .. 2^400,
// was free of overflow and underflow on the way (then x was within 2^+-700)
__device__ __forceinline__ bool in_range(double q) {
  const double a = fabs(q);
  return (a >= 0x1p-300 && a <= 0x1p300) || a == 0.0;
}
__device__ __forceinline__ bool in_range(float q) { return fabsf(q) <= 3.0e38f; }

// A patch's solve with plain divisions, the local vector in `out`: for patches
// whose values leave divide_by's range.  The N lanes r = 0 .. N - 1 of one
// wavefront; its memory operations on one address are ordered once the earlier
// ones are waited for.
template <int N, typename T>
__device__ __attribute__((noinline)) void solve_plain(int m, int ld, const T* L,
                                                      const int32_t* gi, const T* h,
                                                      volatile T* out, int r) {
  for (int i = r; i < m; i += N) out[i] = h[gi[i]];
  __builtin_amdgcn_s_waitcnt(0);
  for (int k = 0; k < m - 1; ++k) {
    const T y = out[k];
    __builtin_amdgcn_s_waitcnt(0);
    for (int i = r; i < m; i += N)
      if (i > k) out[i] = add_rn((T)out[i], -mul_rn(L[k * ld + i], y));
    __builtin_amdgcn_s_waitcnt(0);
  }
  for (int k = m - 1; k >= 0; --k) {
    const T y = (T)out[k] / L[k * ld + k];
    __builtin_amdgcn_s_waitcnt(0);
    for (int i = r; i <= k; i += N)
      out[i] = i == k ? y : add_rn((T)out[i], -mul_rn(L[k * ld + i], y));
    __builtin_amdgcn_s_waitcnt(0);
  }
}

// ------------------------------------------------------------ streamed solve
// Steps U .. 15 of a batch of 16 columns k0 .. k0 + 15 of the forward pass: column
// k updates the rows below k.  HI: the columns are 64 and up (rows lane + 64
// only).  Entries outside the triangle were loaded as zeros and leave their rows
// as they are, so no step needs a condition.
template <bool HI, typename T>
__device__ __forceinline__ void stream_lower(const T (&a0)[16], const T (&a1)[16], int l0, T& v0,
                                             T& v1) {
#pragma unroll
  for (int u = 0; u < 16; ++u) {
    const T y = bcast(HI ? v1 : v0, l0 + u);
    if (!HI) v0 = add_rn(v0, -mul_rn(a0[u], y));
    v1 = add_rn(v1, -mul_rn(a1[u], y));
  }
}

// One wavefront per patch, rows lane and lane + 64, for patches with factors of
// their own.  The column loads of a batch of 16 steps are issued together, before
// the batch's (sequential) updates; each pass reads only its triangle.  Every
// element sees the oracle's operations in its order (divisions: divide_by).  With
// many patches the factors' bytes bound it (13824 patches of 108 unknowns: 310 us
// in FP64, 4.2 TB/s, and 158 in FP32), with few the instructions of the 2 m steps
// and their loads: masks and branches per load and step, a division per step and
// the diagonal in vector registers cost as much again (1728 patches in FP32 41
// instead of 22 us, 13824 in FP64 353).  More batches in flight do not help (4 of
// 8 columns, 2 or 3 of 16: slower, by their registers).
template <typename T>
__global__ __launch_bounds__(kBlock) void k_vanka_solve(int64_t npatches, int m,
                                                        const int32_t* __restrict__ cls, int ld,
                                                        const T* __restrict__ lu,
                                                        const double* __restrict__ rdiag,
                                                        const int32_t* __restrict__ gidx,
                                                        const T* __restrict__ h,
                                                        T* __restrict__ xp) {
  const int lane = threadIdx.x & 63;
  const int64_t p = (int64_t)blockIdx.x * (kBlock / 64) +
                    __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  if (p >= npatches) return;  // the whole wavefront
  const int64_t c = cls[p];
  const T* L = lu + c * ld * m;
  const double* rd = rdiag + c * m;
  // H = P H: gidx holds, per row of the factors, the global entry that the
  // recorded row exchanges bring there
  const int32_t* gi = gidx + p * m;
  const bool in0 = lane < m, in1 = lane + 64 < m;
  T v0 = in0 ? h[gi[lane]] : (T)0;
  T v1 = in1 ? h[gi[lane + 64]] : (T)0;
  const int last = m - 1;
  // Rows and columns past the matrix are zeros (columns past it repeat the last,
  // with y = 0), so only the 16 x 16 blocks on the diagonal need a mask per step;
  // lanes outside a batch's rows leave the loads as a whole.
  // unit lower: column k updates rows i > k
  for (int k0 = 0; k0 < last; k0 += 16) {
    const bool hi = k0 >= 64;
    T a0[16] = {}, a1[16] = {};
    if (!hi && lane >= k0 && lane < ld) {
#pragma unroll
      for (int u = 0; u < 16; ++u) a0[u] = L[(int64_t)min(k0 + u, last) * ld + lane];
    }
    if (lane + 64 >= k0 && lane + 64 < ld) {
#pragma unroll
      for (int u = 0; u < 16; ++u) a1[u] = L[(int64_t)min(k0 + u, last) * ld + lane + 64];
    }
    if (!hi) {
#pragma unroll
      for (int u = 0; u < 16; ++u) a0[u] = lane > k0 + u ? a0[u] : (T)0;
      stream_lower<false>(a0, a1, k0, v0, v1);
    } else {
#pragma unroll
      for (int u = 0; u < 16; ++u) a1[u] = lane + 64 > k0 + u ? a1[u] : (T)0;
      stream_lower<true>(a0, a1, k0 - 64, v0, v1);
    }
  }
  // upper: h_k /= u_kk, then column k updates rows i < k
  for (int k0 = last & ~15; k0 >= 0; k0 -= 16) {
    const bool hi = k0 >= 64;
    T a0[16] = {}, a1[16] = {};
    // lane u keeps column k0 + u's diagonal and its reciprocal
    const int kd = min(k0 + (lane & 15), last);
    const double dl = (double)L[(int64_t)kd * (ld + 1)], rl = rd[kd];
    if (lane < k0 + 16 && lane < ld) {
#pragma unroll
      for (int u = 0; u < 16; ++u) a0[u] = L[(int64_t)min(k0 + u, last) * ld + lane];
    }
    if (hi && lane + 64 < k0 + 16) {
#pragma unroll
      for (int u = 0; u < 16; ++u) a1[u] = L[(int64_t)min(k0 + u, last) * ld + lane + 64];
    }
    if (hi) {
#pragma unroll
      for (int u = 15; u >= 0; --u) {
        const T q = divide_by(v1, lane_read(dl, u), lane_read(rl, u));
        const T y = bcast(q, k0 - 64 + u);
        const T a = lane + 64 < k0 + u ? a1[u] : (T)0;
        v1 = lane + 64 == k0 + u ? q : add_rn(v1, -mul_rn(a, y));
        v0 = add_rn(v0, -mul_rn(a0[u], y));
      }
    } else {
#pragma unroll
      for (int u = 15; u >= 0; --u) {
        const T q = divide_by(v0, lane_read(dl, u), lane_read(rl, u));
        const T y = bcast(q, k0 + u);
        const T a = lane < k0 + u ? a0[u] : (T)0;
        v0 = lane == k0 + u ? q : add_rn(v0, -mul_rn(a, y));
      }
    }
  }
  T* out = xp + p * (int64_t)m;
  const bool ok = (!in0 || (in_range(v0) && rd[lane] != 0.0)) &&
                  (!in1 || (in_range(v1) && rd[lane + 64] != 0.0));
  if (__builtin_expect(__ballot(!ok) != 0, 0)) {
    solve_plain<64>(m, ld, L, gi, h, out, lane);
    return;
  }
  if (in0) out[lane] = v0;
  if (in1) out[lane + 64] = v1;
}

// ------------------------------------------------------------- grouped solve
// lane N of each 16-lane row, to the whole row
template <int N>
__device__ __forceinline__ float row_bcast(float x) {
  const int b = __builtin_bit_cast(int, x);
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(b, b, 0x150 + N, 0xf, 0xf, false));
}
template <int N>
__device__ __forceinline__ double row_bcast(double x) {
  const int64_t b = __builtin_bit_cast(int64_t, x);
  const int l = (int)(b & 0xFFFFFFFF), h = (int)(b >> 32);
  const int lo = __builtin_amdgcn_update_dpp(l, l, 0x150 + N, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(h, h, 0x150 + N, 0xf, 0xf, false);
  return __builtin_bit_cast(double, ((int64_t)hi << 32) | (uint32_t)lo);
}

// The passes go in sets of kSet columns: the next set's factors are read from
// LDS before this set's steps, and no read or address moves further (the
// compiler would otherwise hoist all of them and spill).  v[j] is the lane's
// row 16 j + r, r = lane % 16.
template <typename T> constexpr int kSet = sizeof(T) == 8 ? 2 : 4;
__device__ __forceinline__ void reads_stay(int& r) {
  asm volatile("" : "+v"(r)::"memory");
  __builtin_amdgcn_sched_barrier(0);
}

// columns S kSet .. S kSet + kSet - 1, rows from the diagonal's 16 down
template <int MB, int S, typename T>
__device__ __forceinline__ void load_lower(const T* __restrict__ L, int r, T (&c)[kSet<T>][MB]) {
#pragma unroll
  for (int s = 0; s < kSet<T>; ++s) {
    const int k = S * kSet<T> + s;
#pragma unroll
    for (int j = k / 16; j < MB; ++j) c[s][j] = L[r + k * 16 * MB + 16 * j];
  }
}
// forward step (unit lower triangle): column k updates the rows below k
template <int MB, int K, typename T>
__device__ __forceinline__ void step_lower(const T (&c)[MB], int r, T (&v)[MB]) {
  constexpr int KB = K / 16, N = K % 16;
  const T y = row_bcast<N>(v[KB]);
  if constexpr (N < 15) {
    const T u = add_rn(v[KB], -mul_rn(c[KB], y));
    v[KB] = r > N ? u : v[KB];
  }
#pragma unroll
  for (int j = KB + 1; j < MB; ++j) v[j] = add_rn(v[j], -mul_rn(c[j], y));
}
template <int MB, int S, typename T>
__device__ __forceinline__ void group_forward(const T* __restrict__ L, int r, T (&v)[MB],
                                              const T (&c)[kSet<T>][MB]) {
  constexpr int Q = kSet<T>, K = S * Q;
  T next[Q][MB];
  if constexpr (K + Q < 16 * MB) load_lower<MB, S + 1>(L, r, next);
  reads_stay(r);
  step_lower<MB, K>(c[0], r, v);
  step_lower<MB, K + 1>(c[1], r, v);
  if constexpr (Q == 4) {
    step_lower<MB, K + 2>(c[2], r, v);
    step_lower<MB, K + 3>(c[3], r, v);
  }
  if constexpr (K + Q < 16 * MB) group_forward<MB, S + 1>(L, r, v, next);
}

template <typename T, int MB>
struct UpperSet {
  T c[kSet<T>][MB];
  double d[kSet<T>], rk[kSet<T>];  // u_kk and its reciprocal
};
// columns S kSet .. S kSet + kSet - 1, rows up to the diagonal's 16
template <int MB, int S, typename T>
__device__ __forceinline__ void load_upper(const T* __restrict__ L, int r,
                                           const double* __restrict__ rd, UpperSet<T, MB>& u) {
#pragma unroll
  for (int s = 0; s < kSet<T>; ++s) {
    const int k = S * kSet<T> + s;
#pragma unroll
    for (int j = 0; j <= k / 16; ++j) u.c[s][j] = L[r + k * 16 * MB + 16 * j];
    u.d[s] = rd[2 * k];
    u.rk[s] = rd[2 * k + 1];
  }
}
// backward step: y_k = v_k / u_kk, then column k updates the rows above k.
// Rows and columns past the matrix are zeros in LDS (u_kk = 1) and stay zero.
template <int MB, int K, typename T>
__device__ __forceinline__ void step_upper(const T (&c)[MB], double d, double rk, int r,
                                           T (&v)[MB]) {
  constexpr int KB = K / 16, N = K % 16;
  const T q = divide_by(v[KB], d, rk);
  const T y = row_bcast<N>(q);
  const T u = add_rn(v[KB], -mul_rn(c[KB], y));
  v[KB] = r < N ? u : (r == N ? q : v[KB]);
#pragma unroll
  for (int j = 0; j < KB; ++j) v[j] = add_rn(v[j], -mul_rn(c[j], y));
}
template <int MB, int S, typename T>
__device__ __forceinline__ void group_backward(const T* __restrict__ L,
                                               const double* __restrict__ rd, int r,
                                               T (&v)[MB], const UpperSet<T, MB>& u) {
  constexpr int Q = kSet<T>, K = S * Q;
  UpperSet<T, MB> next;
  if constexpr (S > 0) load_upper<MB, S - 1>(L, r, rd, next);
  reads_stay(r);
  if constexpr (Q == 4) {
    step_upper<MB, K + 3>(u.c[3], u.d[3], u.rk[3], r, v);
    step_upper<MB, K + 2>(u.c[2], u.d[2], u.rk[2], r, v);
  }
  step_upper<MB, K + 1>(u.c[1], u.d[1], u.rk[1], r, v);
  step_upper<MB, K>(u.c[0], u.d[0], u.rk[0], r, v);
  if constexpr (S > 0) group_backward<MB, S - 1>(L, rd, r, v, next);
}

// entries of T the grouped solve keeps in LDS: the columns, 16 MB rows each,
// zeros up to column 16 MB
__host__ __device__ constexpr int group_entries(int mb) { return 256 * mb * mb; }

// Patches of one class per workgroup: the factors go to LDS once (16-byte
// loads, the first local vectors gathered meanwhile), then 16 lanes solve each
// patch, lane r holding its rows r, r + 16, ... (MB of them), the solved value
// broadcast to the 16 lanes by one DPP move per half.  A wavefront thus solves 4
// patches at a time with the LDS reads shared between them; every entry sees the
// operations of k_vanka_solve in the same order.  Bound by the chain of 2 m
// dependent steps while a CU has few patches, then by their LDS reads and issue,
// not by memory: 108 unknowns, 68 classes, 512 patches 13.9 us in FP32 and 17.4 in
// FP64 (one wavefront and one set of factors per patch 36 and 40), 4096 18.6 and
// 26.6 (56 and 107), 32768 60 and 105.
constexpr int kGroupThreads = 512;
template <typename T, int MB>
__global__ __launch_bounds__(kGroupThreads) void k_vanka_group(int m, int64_t lstride,
                                                     const T* __restrict__ lu,
                                                     const double* __restrict__ rdiag,
                                                     const int32_t* __restrict__ groups,
                                                     const int32_t* __restrict__ plist,
                                                     const int32_t* __restrict__ gidx,
                                                     const T* __restrict__ h,
                                                     T* __restrict__ xp) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ double rd[32 * MB];  // u_kk and its reciprocal
  T* L = reinterpret_cast<T*>(smem);
  const int32_t* g = groups + 3 * (int64_t)blockIdx.x;
  const int64_t c = g[0], first = g[1];
  const int count = g[2];
  int r = threadIdx.x & 15;
  int t = threadIdx.x >> 4;
  T v[MB];
  auto gather = [&]() {
    const int32_t* gi = gidx + (int64_t)plist[first + t] * m;
#pragma unroll
    for (int j = 0; j < MB; ++j) v[j] = (16 * j + r < m) ? h[gi[16 * j + r]] : (T)0;
  };
  if (t < count) gather();  // in flight while the factors are staged
  typedef int v4 __attribute__((ext_vector_type(4)));
  constexpr int per = 16 / sizeof(T);
  const v4* src = reinterpret_cast<const v4*>(lu + c * lstride);
  v4* dst = reinterpret_cast<v4*>(smem);
  const int n16 = 16 * MB * m / per, all16 = group_entries(MB) / per;
  // up to 8 loads in flight per thread
  for (int e0 = threadIdx.x; e0 < n16; e0 += 8 * kGroupThreads) {
    v4 x[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int e = e0 + u * kGroupThreads;
      x[u] = e < n16 ? src[e] : v4{0, 0, 0, 0};
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int e = e0 + u * kGroupThreads;
      if (e < n16) dst[e] = x[u];
    }
  }
  for (int e = n16 + threadIdx.x; e < all16; e += kGroupThreads) dst[e] = v4{0, 0, 0, 0};
  bool plain = false;  // a zero or extreme diagonal
  for (int k = threadIdx.x; k < 16 * MB; k += kGroupThreads) {
    rd[2 * k] = k < m ? (double)lu[c * lstride + k * (16 * MB + 1)] : 1.0;
    rd[2 * k + 1] = k < m ? rdiag[c * m + k] : 1.0;
    plain = rd[2 * k + 1] == 0.0;
  }
  plain = __syncthreads_or(plain);
  for (; t < count;) {
    reads_stay(r);
    {
      T c[kSet<T>][MB];
      load_lower<MB, 0>(L, r, c);
      group_forward<MB, 0>(L, r, v, c);
    }
    {
      constexpr int last = 16 * MB / kSet<T> - 1;
      UpperSet<T, MB> u;
      load_upper<MB, last>(L, r, rd, u);
      group_backward<MB, last>(L, rd, r, v, u);
    }
    const int64_t p = plist[first + t];
    T* out = xp + p * (int64_t)m;
    bool ok = !plain;
#pragma unroll
    for (int j = 0; j < MB; ++j) ok = ok && in_range(v[j]);
    const uint64_t bad = __ballot(!ok) >> (threadIdx.x & 48);
    if (__builtin_expect((bad & 0xFFFF) != 0, 0)) {
      solve_plain<16>(m, 16 * MB, lu + c * lstride, gidx + p * m, h, out, r);
    } else {
#pragma unroll
      for (int j = 0; j < MB; ++j)
        if (16 * j + r < m) out[16 * j + r] = v[j];
    }
    t += kGroupThreads / 16;
    if (t < count) gather();
  }
}

// h(i, c) = (sum over the patches of node i, ascending) * (1 / count_i); mode 0
// x = h, 1 x += omega h (StdSolver::smooth), 2 x = omega h
template <typename T>
__global__ __launch_bounds__(kBlock) void k_vanka_average(int64_t n, int B, int psize, int m,
                                                          const int32_t* __restrict__ nptr,
                                                          const int32_t* __restrict__ nent,
                                                          const T* __restrict__ xp,
                                                          T* __restrict__ x, int mode, T omega) {
  const int64_t t = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (t >= n * B) return;
  const int64_t i = t / B;
  const int c = (int)(t - i * B);
  const int32_t e0 = nptr[i], e1 = nptr[i + 1];
  T acc = (T)0;
  for (int32_t e = e0; e < e1; ++e) {
    const int32_t pe = nent[e];
    const int64_t pp = pe / psize;
    const int r = pe - (int)(pp * psize);
    acc = add_rn(acc, xp[pp * m + B * r + c]);
  }
  const double s = 1.0 / (double)(e1 - e0);
  const T h = (T)mul_rn((double)acc, s);
  if (mode == 0)
    x[t] = h;
  else if (mode == 1)
    x[t] = add_rn(x[t], mul_rn(omega, h));
  else
    x[t] = mul_rn(omega, h);
}

template <typename T, int MB>
int group_launch(gh_ctx* ctx, const gh_vanka* V, const T* h) {
  const int lds = group_entries(MB) * (int)sizeof(T);
  hipLaunchKernelGGL((k_vanka_group<T, MB>), dim3((unsigned)V->ngroups), dim3(kGroupThreads), lds,
                     ctx->stream, V->m, V->lstride, (const T*)V->lu, V->rdiag, V->groups, V->plist,
                     V->piv, h, (T*)V->xp);
  GH_HIP(hipGetLastError());
  return GH_OK;
}

// Workgroups of the grouped solve for local systems of m unknowns that a CU holds
// at once (LDS, registers and wavefronts; 0: none); their LDS is allowed here.
template <typename T>
int group_fit(int m) {
  const int mb = (m + 15) / 16;
  const void* k[8] = {(const void*)k_vanka_group<T, 1>, (const void*)k_vanka_group<T, 2>,
                      (const void*)k_vanka_group<T, 3>, (const void*)k_vanka_group<T, 4>,
                      (const void*)k_vanka_group<T, 5>, (const void*)k_vanka_group<T, 6>,
                      (const void*)k_vanka_group<T, 7>, (const void*)k_vanka_group<T, 8>};
  const int lds = group_entries(mb) * (int)sizeof(T);
  int fit = 0;
  if (hipFuncSetAttribute(k[mb - 1], hipFuncAttributeMaxDynamicSharedMemorySize, lds) == hipSuccess &&
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&fit, k[mb - 1], kGroupThreads, lds) == hipSuccess)
    return fit;
  (void)hipGetLastError();
  return 0;
}

template <typename T>
int vanka_apply_t(gh_ctx* ctx, const gh_vanka* V, const T* in, T* out, int mode, T omega) {
  if (V->ngroups > 0) {
    int rc = GH_OK;
    switch ((V->m + 15) / 16) {
      case 1: rc = group_launch<T, 1>(ctx, V, in); break;
      case 2: rc = group_launch<T, 2>(ctx, V, in); break;
      case 3: rc = group_launch<T, 3>(ctx, V, in); break;
      case 4: rc = group_launch<T, 4>(ctx, V, in); break;
      case 5: rc = group_launch<T, 5>(ctx, V, in); break;
      case 6: rc = group_launch<T, 6>(ctx, V, in); break;
      case 7: rc = group_launch<T, 7>(ctx, V, in); break;
      default: rc = group_launch<T, 8>(ctx, V, in); break;
    }
    GH_TRY(rc);
  } else {
    const unsigned gs = (unsigned)((V->npatches + kBlock / 64 - 1) / (kBlock / 64));
    hipLaunchKernelGGL(k_vanka_solve<T>, dim3(gs), dim3(kBlock), 0, ctx->stream, V->npatches,
                       V->m, V->cls, V->ld, (const T*)V->lu, V->rdiag, V->piv, in, (T*)V->xp);
  }
  const unsigned ga = (unsigned)((V->n * V->B + kBlock - 1) / kBlock);
  hipLaunchKernelGGL(k_vanka_average<T>, dim3(ga), dim3(kBlock), 0, ctx->stream, V->n, V->B,
                     V->psize, V->m, V->nptr, V->nent, (const T*)V->xp, out, mode, omega);
  GH_HIP(hipGetLastError());
  return GH_OK;
}

// The first patch with each patch's matrix, by hash (`first`; the entries are
// compared afterwards, k_vanka_same).  scratch: 2 * npatches 64-bit words.
int patch_firsts(gh_ctx* ctx, const gh_csr* A, int64_t npatches, int psize, int B,
                 const int32_t* d_nodes, void* scratch, std::vector<int32_t>& first) {
  const size_t lds = sizeof(int32_t) * (size_t)psize * psize;
  uint64_t* d_hash = (uint64_t*)scratch;
  std::vector<uint64_t> hash(2 * npatches);
  GH_HIP(hipFuncSetAttribute((const void*)k_vanka_hash,
                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  hipLaunchKernelGGL(k_vanka_hash, dim3((unsigned)npatches), dim3(kHashThreads), lds, ctx->stream,
                     psize, B, d_nodes, A->rowptr, A->col, (const double*)A->val, d_hash);
  GH_HIP(hipGetLastError());
  GH_HIP(hipMemcpyAsync(hash.data(), d_hash, sizeof(uint64_t) * hash.size(), hipMemcpyDeviceToHost,
                        ctx->stream));
  GH_HIP(hipStreamSynchronize(ctx->stream));
  KeyTable table(npatches, -1);
  first.resize(npatches);
  for (int64_t p = 0; p < npatches; ++p) {
    int64_t& f = table[hash[2 * p] ^ (hash[2 * p + 1] * 0x9E3779B97F4A7C15ull)];
    if (f < 0) f = p;
    first[p] = (int32_t)f;
  }
  return GH_OK;
}

// The patches by class: cls[p], and reps[c] the first patch of class c (classes
// in order of first appearance).  A patch that differs from its first has a class
// of its own.
void patch_classes(const std::vector<int32_t>& first, const std::vector<int32_t>& differs,
                   std::vector<int32_t>& cls, std::vector<int32_t>& reps) {
  cls.assign(first.size(), -1);
  reps.clear();
  for (size_t p = 0; p < first.size(); ++p) {  // first[p] <= p
    if (first[p] == (int32_t)p || differs[p]) {
      cls[p] = (int32_t)reps.size();
      reps.push_back((int32_t)p);
    } else {
      cls[p] = cls[first[p]];
    }
  }
}

// Whether the grouped solve runs, and its groups: chunks of a class's patches, as
// many per workgroup as make the solve shortest.  A CU works off its share of the
// workgroups, `fit` at a time; they take their patches' LDS reads and issue one
// after the other, with the staging on top, but not less than the chain of 2 m
// steps, which is as long as the work of 24 patches at m = 108 and of more where a
// patch is smaller.  108 unknowns, FP64 (FP32), copy and averaging included: 32768
// patches in 68 classes, 72 to a workgroup 124 us (75), 128 187 (109), 32 147 (74),
// 8 292 (103); 4096 patches, 20 to a workgroup 36 (26), 8 61 (28), 64 55 (39).
//
// Against the streamed solve the groups must hold enough patches for the factors
// staged: with one patch each they are slower for any number of patches (108
// unknowns, 64 patches 24.3 against 23.6 us in FP64; 512 in FP32 27.4 against
// 22.0), with two where a wavefront of the streamed solve has no second row per
// lane (m <= 64: 2048 patches of 36, FP64, 13.4 against 16.9; 81 unknowns, FP32,
// 25.6 against 22.3), with three beyond (108, 512 patches, 21.3 against 27.5).  Once
// the workgroups come in rounds, a CU that holds few of them waits for their
// staging, so there it is patches per place of a CU: 108 unknowns in FP64 (one
// workgroup per CU), 2048 patches in classes of 2, 3, 4, 5 and 8: 83, 59, 43, 42 and
// 25 us against 40, 44, 38, 44 and 38; 81 unknowns (two per CU), 8192 patches in
// classes of 2, 3, 4: 139, 103, 76 against 106, 102, 100; 54 unknowns, classes of 2:
// 54 against 59.
void vanka_groups(gh_ctx* ctx, gh_vanka* V, const std::vector<int32_t>& cls,
                  std::vector<int32_t>& plist, std::vector<int32_t>& groups) {
  const int64_t np = V->npatches, nc = V->nclasses;
  const int64_t fit = V->prec == GH_F64 ? group_fit<double>(V->m) : group_fit<float>(V->m);
  if (fit < 1) return;
  const int64_t at_once = fit * ctx->num_cu;
  std::vector<int64_t> start(nc + 1, 0);
  for (int64_t p = 0; p < np; ++p) start[cls[p] + 1]++;
  const int64_t most = *std::max_element(start.begin(), start.end());
  const int64_t least = V->m > 64 ? 3 : 2;  // patches per group
  const int64_t cu = ctx->num_cu;
  const double stage = 8.0, chain = 24.0 * 108.0 / V->m;  // in patches
  auto time = [&](int64_t groups, int64_t c) {  // of the CU that has the most groups
    const int64_t share = (groups + cu - 1) / cu, full = share / fit, rest = share % fit;
    return (double)full * std::max(chain, (double)(fit * c) + stage) +
           (rest ? std::max(chain, (double)(rest * c) + stage) : 0.0);
  };
  int64_t chunk = 0, ng = 0;
  double best = 0.0;
  for (int64_t c = 4;; c += 4) {  // a wavefront takes 4 patches
    int64_t g = 0;
    for (int64_t k = 1; k <= nc; ++k) g += (start[k] + c - 1) / c;
    const double cost = time(g, c);
    if (chunk == 0 || cost < best || (cost == best && np < least * ng)) {
      chunk = c;
      ng = g;
      best = cost;
    }
    // one group per class is the least there can be
    if (c >= most || time(nc, c) > best) break;
  }
  if (np < least * ng || (ng > at_once && np * fit < (least + 2) * ng)) return;
  for (int64_t c = 0; c < nc; ++c) start[c + 1] += start[c];
  plist.resize(np);
  {
    std::vector<int64_t> fill(start.begin(), start.end() - 1);
    for (int64_t p = 0; p < np; ++p) plist[fill[cls[p]]++] = (int32_t)p;
  }
  for (int64_t c = 0; c < nc; ++c)
    for (int64_t a = start[c]; a < start[c + 1]; a += chunk) {
      groups.push_back((int32_t)c);
      groups.push_back((int32_t)a);
      groups.push_back((int32_t)std::min(chunk, start[c + 1] - a));
    }
  V->ngroups = (int64_t)groups.size() / 3;
}

}  // namespace

namespace gh {

int vanka_apply(gh_ctx* ctx, const gh_vanka* V, int prec, const void* in, void* out, int mode,
                double omega) {
  if (prec != V->prec) return fail(GH_EINVAL, "vanka: vector precision differs from the factors'");
  if (V->npatches == 0) return GH_OK;
  if (prec == GH_F64)
    return vanka_apply_t<double>(ctx, V, (const double*)in, (double*)out, mode, omega);
  return vanka_apply_t<float>(ctx, V, (const float*)in, (float*)out, mode, (float)omega);
}

int vanka_create(gh_ctx* ctx, const gh_csr* A, int64_t npatches, int psize, const int32_t* nodes,
                 int prec, gh_vanka** out) {
  GH_ARG(ctx && A && out && (nodes || npatches == 0) && npatches >= 0 && psize >= 1,
         "gh_vanka_create: bad arguments");
  GH_ARG(A->prec == GH_F64, "gh_vanka_create: the matrix must be FP64");
  GH_ARG(prec == GH_F64 || prec == GH_F32, "gh_vanka_create: factors are FP64 or FP32");
  const int B = A->ncomp, m = psize * B;
  GH_ARG(psize <= kVankaMaxNodes && m <= kVankaMaxM,
         "gh_vanka_create: at most 128 unknowns per patch");
  GH_ARG(A->nnz > 0 || npatches == 0, "gh_vanka_create: patches of a matrix without entries");
  const int64_t n = A->n;
  // node -> (patch, local) lists, ascending patch; every node must be covered
  std::vector<int32_t> nptr(n + 1, 0), nent((size_t)npatches * psize);
  for (int64_t k = 0; k < npatches * psize; ++k) {
    if (nodes[k] < 0 || nodes[k] >= n) return fail(GH_EINVAL, "gh_vanka_create: node out of range");
    nptr[nodes[k] + 1]++;
  }
  for (int64_t p = 0; p < npatches; ++p)
    for (int r = 0; r < psize; ++r)
      for (int t = 0; t < r; ++t)
        if (nodes[p * psize + t] == nodes[p * psize + r])
          return fail(GH_EINVAL, "gh_vanka_create: patch %lld lists a node twice", (long long)p);
  for (int64_t i = 0; i < n; ++i) {
    if (nptr[i + 1] == 0) return fail(GH_EINVAL, "gh_vanka_create: node %lld is in no patch", (long long)i);
    nptr[i + 1] += nptr[i];
  }
  {
    std::vector<int32_t> fill(nptr.begin(), nptr.end() - 1);
    for (int64_t p = 0; p < npatches; ++p)
      for (int r = 0; r < psize; ++r) nent[fill[nodes[p * psize + r]]++] = (int32_t)(p * psize + r);
  }
  gh_vanka* V = new gh_vanka();
  V->ctx = ctx;
  ctx_retain(ctx);
  V->B = B;
  V->psize = psize;
  V->m = m;
  V->prec = prec;
  V->n = n;
  V->npatches = npatches;
  auto bail = [&](int rc) {
    gh_vanka_destroy(V);
    return rc;
  };
  // Few allocations and copies, since they are most of what the creation of a small
  // level costs (64 patches of 108: 0.26 ms).  ints: nodes, nptr, nent; then per
  // factorisation cls, reps; then the gather, plist and groups.
  const size_t ts = prec == GH_F64 ? 8 : 4;
  const int64_t np = npatches, ne = np * psize;
  if (hipMalloc((void**)&V->ints, sizeof(int32_t) * (2 * ne + (n + 1) + np * (m + 6))) != hipSuccess ||
      hipMalloc(&V->xp, std::max<size_t>({ts * np * m, sizeof(int32_t) * np * (m + 2),
                                          sizeof(uint64_t) * 2 * np, 8})) != hipSuccess)
    return bail(fail(GH_ENOMEM, "gh_vanka_create: allocation failed"));
  V->nodes = V->ints;
  V->nptr = V->nodes + ne;
  V->nent = V->nptr + n + 1;
  V->cls = V->nent + ne;
  int32_t* d_reps = V->cls + np;
  V->piv = d_reps + np;
  V->plist = V->piv + np * m;
  V->groups = V->plist + np;  // at most one per patch
  {
    std::vector<int32_t> up(2 * ne + n + 1);
    std::copy(nodes, nodes + ne, up.begin());
    std::copy(nptr.begin(), nptr.end(), up.begin() + ne);
    std::copy(nent.begin(), nent.end(), up.begin() + ne + n + 1);
    if (hipMemcpy(V->nodes, up.data(), sizeof(int32_t) * up.size(), hipMemcpyHostToDevice) != hipSuccess)
      return bail(fail(GH_EHIP, "gh_vanka_create: upload failed"));
  }
  if (npatches > 0) {
    std::vector<int32_t> first, cls, reps, piv, differs(np, 0);
    if (int rc = patch_firsts(ctx, A, np, psize, B, V->nodes, V->xp, first)) return bail(rc);
    V->ld = (m + 15) / 16 * 16;
    V->lstride = (int64_t)V->ld * m;
    const size_t lds = sizeof(int32_t) * (size_t)psize * psize;
    // Factors of the classes, and beside them the comparison of the patches with
    // their firsts; hashes that agreed by chance make one more turn.
    auto factor = [&]() -> int {
      const int64_t nc = V->nclasses = (int64_t)reps.size();
      const size_t lub = ts * nc * V->lstride;
      if (V->lu) (void)hipFree(V->lu);
      V->lu = nullptr;
      if (hipMalloc(&V->lu, lub + sizeof(double) * nc * m) != hipSuccess)
        return fail(GH_ENOMEM, "gh_vanka_create: allocation failed");
      V->rdiag = (double*)((char*)V->lu + lub);
      int32_t *d_piv = (int32_t*)V->xp, *d_first = d_piv + nc * m, *d_differs = d_first + np;
      std::vector<int32_t> up(cls);
      up.insert(up.end(), reps.begin(), reps.end());
      GH_HIP(hipMemcpyAsync(V->cls, up.data(), sizeof(int32_t) * up.size(), hipMemcpyHostToDevice,
                            ctx->stream));
      GH_HIP(hipFuncSetAttribute((const void*)k_vanka_factor,
                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
      hipLaunchKernelGGL(k_vanka_factor, dim3((unsigned)nc), dim3(kFactorThreads), lds, ctx->stream,
                         psize, B, d_reps, V->nodes, A->rowptr, A->col, (const double*)A->val,
                         V->ld, prec == GH_F64 ? (double*)V->lu : nullptr,
                         prec == GH_F64 ? nullptr : (float*)V->lu, d_piv);
      GH_HIP(hipGetLastError());
      const dim3 gr((unsigned)((nc * m + kBlock - 1) / kBlock));
      if (prec == GH_F64)
        hipLaunchKernelGGL(k_vanka_rdiag<double>, gr, dim3(kBlock), 0, ctx->stream, nc, m,
                           V->ld, (const double*)V->lu, V->rdiag);
      else
        hipLaunchKernelGGL(k_vanka_rdiag<float>, gr, dim3(kBlock), 0, ctx->stream, nc, m,
                           V->ld, (const float*)V->lu, V->rdiag);
      GH_HIP(hipGetLastError());
      const bool compare = nc < np;
      if (compare) {
        GH_HIP(hipMemcpyAsync(d_first, first.data(), sizeof(int32_t) * np, hipMemcpyHostToDevice,
                              ctx->stream));
        GH_HIP(hipFuncSetAttribute((const void*)k_vanka_same,
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)(2 * lds)));
        hipLaunchKernelGGL(k_vanka_same, dim3((unsigned)np), dim3(kHashThreads), 2 * lds, ctx->stream,
                           psize, B, V->nodes, A->rowptr, A->col, (const double*)A->val, d_first,
                           d_differs);
        GH_HIP(hipGetLastError());
      }
      piv.resize((size_t)nc * m + (compare ? 2 * np : 0));
      GH_HIP(hipMemcpyAsync(piv.data(), d_piv, sizeof(int32_t) * piv.size(), hipMemcpyDeviceToHost,
                            ctx->stream));
      GH_HIP(hipStreamSynchronize(ctx->stream));
      return GH_OK;
    };
    for (;;) {
      patch_classes(first, differs, cls, reps);
      if (int rc = factor()) return bail(rc);
      const int64_t nc = V->nclasses;
      if (nc == np || std::equal(differs.begin(), differs.end(), piv.begin() + nc * m + np)) break;
      differs.assign(piv.begin() + nc * m + np, piv.end());
    }
    const int64_t nc = V->nclasses;
    // Compose the recorded row exchanges (applied in order k = 0..m-1) into
    // one gather: row i of P h is local entry src[i], i.e. the global entry
    // node(src[i] / B) * B + src[i] % B.  The solve then needs no exchanges.
    std::vector<int32_t> src((size_t)nc * m), lists((size_t)np * m), plist, groups;
    for (int64_t c = 0; c < nc; ++c) {
      const int32_t* pv = piv.data() + c * m;
      int32_t* sc = src.data() + c * m;
      for (int i = 0; i < m; ++i) sc[i] = i;
      for (int k = 0; k < m; ++k) {
        if (pv[k] < k || pv[k] >= m) return bail(fail(GH_EINVAL, "gh_vanka_create: bad pivot"));
        std::swap(sc[k], sc[pv[k]]);
      }
    }
    parallel_for(np, 2048, [&](int64_t a, int64_t b) {
      for (int64_t p = a; p < b; ++p) {
        const int32_t* sc = src.data() + (int64_t)cls[p] * m;
        for (int i = 0; i < m; ++i)
          lists[p * m + i] = (int32_t)((int64_t)nodes[p * psize + sc[i] / B] * B + sc[i] % B);
      }
    });
    vanka_groups(ctx, V, cls, plist, groups);
    lists.insert(lists.end(), plist.begin(), plist.end());
    lists.insert(lists.end(), groups.begin(), groups.end());
    if (hipMemcpy(V->piv, lists.data(), sizeof(int32_t) * lists.size(), hipMemcpyHostToDevice) != hipSuccess)
      return bail(fail(GH_EHIP, "gh_vanka_create: gather upload failed"));
  }
  *out = V;
  return GH_OK;
}

}  // namespace gh

extern "C" {

int gh_vanka_create(gh_ctx* ctx, const gh_csr* A, int64_t npatches, int psize,
                    const int32_t* nodes, int prec, gh_vanka** out) {
  GH_ARG(A, "gh_vanka_create: NULL matrix");
  GH_ARG(!A->host_only, "gh_vanka_create: the matrix has no device layout (created by gh_csr_create_host)");
  return vanka_create(ctx, A, npatches, psize, nodes, prec, out);
}

int gh_vanka_destroy(gh_vanka* V) {
  if (!V) return GH_OK;
  if (V->ctx && V->ctx->stream) (void)hipStreamSynchronize(V->ctx->stream);
  for (void* p : {(void*)V->ints, V->lu, V->xp})
    if (p) (void)hipFree(p);
  gh_ctx* ctx = V->ctx;
  delete V;
  if (ctx) ctx_release(ctx);
  return GH_OK;
}

int64_t gh_vanka_groups(const gh_vanka* V) { return V ? V->ngroups : 0; }

int gh_vanka_solve(gh_ctx* ctx, const gh_vanka* V, gh_vec* x) {
  GH_ARG(ctx && V && x, "gh_vanka_solve: NULL argument");
  GH_ARG(x->n == V->n && x->ncomp == V->B, "gh_vanka_solve: vector shape does not match");
  return vanka_apply(ctx, V, x->prec, x->d, x->d, 0, 1.0);
}

}  // extern "C"
