// Direct solve of the coarsest multigrid levels: the dense inverse of the
// level matrix, formed on the device (Gauss-Jordan with partial pivoting in
// panels of 32 columns for scalar levels of up to 1024 unknowns; else LU with
// partial pivoting and the inverse from it, rocSOLVER getrf / getri) and applied by k_dense_solve.
// The reference solves its coarse level with UMFPACK when it is built with it
// (src/LinAlg/umfilu.cc, StdSolver::DirectSolver) and otherwise with
// iterexact smoothing sweeps; any exact solve gives the same V-cycle up to
// rounding.
#include <rocblas/rocblas.h>
#include <rocsolver/rocsolver.h>

#include <algorithm>
#include <climits>

#include "gh_kernels.h"

using namespace gh;

namespace {

// dense[i * m + j] = A(i, j) (row-major, zero before), node blocks expanded; one
// wavefront per block row (a row's columns are distinct)
__global__ __launch_bounds__(kBlock) void k_scatter_dense(int64_t n, int B, int64_t m,
                                                          const int32_t* __restrict__ rowptr,
                                                          const int32_t* __restrict__ col,
                                                          const double* __restrict__ val,
                                                          double* __restrict__ dense) {
  const int64_t i = (int64_t)blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
  if (i >= n) return;
  const int BB = B * B;
  for (int32_t pos = rowptr[i] + (threadIdx.x & 63); pos < rowptr[i + 1]; pos += 64) {
    const int64_t j = col[pos];
    for (int r = 0; r < B; ++r)
      for (int c = 0; c < B; ++c)
        dense[(i * B + r) * m + j * B + c] = val[(int64_t)pos * BB + r * B + c];
  }
}

// ------------------------------------------------------ Gauss-Jordan inverse
// In place of A (m x m, row-major), panel by panel of kPanel columns, without
// moving rows: column j takes its pivot in row p_j, the row of largest |a_ij|
// (the first of them) among those no column has taken.  After the last panel
// entry (p_j, i) is entry (j, p_i) of the inverse.
//   k_gj_panel  one workgroup, two rows per thread: the panel's columns of the
//               transformation (rows in registers, the pivot row through LDS),
//   k_gj_update all other columns at once: a rank-kPanel product, out of place,
//               so that every workgroup may read the pivot rows.
// Bound by the chain of m pivot steps (2.2 us each at m = 729: search, exchange,
// one pass over the panel's rows; the updates are 11 us per panel).  The direct
// levels of a 64^3 hierarchy (27, 125, 729 unknowns) take 2.6 ms, with rocSOLVER's
// LU and inverse 5.1.
constexpr int kPanel = 32;
constexpr int kGjThreads = 512;  // of a panel, kGjRows rows each
constexpr int kGjRows = 2;
constexpr int kGjMax = kGjThreads * kGjRows;  // unknowns
constexpr int kTileRows = 32, kTileCols = 64;  // update: entries per workgroup of 256

// columns k0 .. k0 + w - 1 (w <= kPanel): W (kPanel x m) receives the panel,
// piv[k0 + t] the pivot rows; taken[row] is k0 + 1 for the rows that got a pivot
// here.  flag: the first column whose candidates are zeros, plus one (NaNs among
// them are no zeros: the inverse is then NaN, as from an LU).
// A thread's rows turn by one register per column, so that the column in hand is
// always a[.][0] and the loop stays small.
__global__ __launch_bounds__(kGjThreads) void k_gj_panel(int m, int k0, int w,
                                                         const double* __restrict__ A,
                                                         double* __restrict__ W,
                                                         int32_t* __restrict__ piv,
                                                         int32_t* __restrict__ taken, int* flag) {
  __shared__ double prow[2][kPanel];           // the scaled pivot row; entry 0: 1 / pivot
  __shared__ double sbest[2][kGjThreads / 64];  // per wavefront: the largest candidate
  __shared__ int srow[2][kGjThreads / 64];      // and its row
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  double a[kGjRows][kPanel];
  bool free_row[kGjRows];
  int row[kGjRows];
#pragma unroll
  for (int g = 0; g < kGjRows; ++g) {
    row[g] = threadIdx.x + g * blockDim.x;
    free_row[g] = row[g] < m && taken[row[g]] == 0;
#pragma unroll
    for (int t = 0; t < kPanel; ++t)
      a[g][t] = (row[g] < m && t < w) ? A[(int64_t)row[g] * m + k0 + t] : 0.0;
  }
#pragma unroll 1
  for (int t = 0; t < w; ++t) {
    const int buf = t & 1;
    // the largest |a_it| of the free rows (a NaN is passed over), then the first
    // row holding it; with no number among them the first free row
    double best = 0.0;
#pragma unroll
    for (int g = 0; g < kGjRows; ++g)
      best = fmax(best, free_row[g] ? fabs(a[g][0]) : 0.0);  // fmax passes NaN over
    best = wave_max_nonneg(best);
    int first = INT_MAX;
#pragma unroll
    for (int g = 0; g < kGjRows; ++g)
      if (free_row[g] && fabs(a[g][0]) == best) first = min(first, row[g]);
    first = wave_min(first);
    if (first == INT_MAX) {  // no free row here, or NaNs only
#pragma unroll
      for (int g = 0; g < kGjRows; ++g)
        if (free_row[g]) first = min(first, row[g]);
      first = wave_min(first);
      best = first == INT_MAX ? -2.0 : -1.0;
    }
    if (lane == 0) {
      sbest[buf][wave] = best;
      srow[buf][wave] = first;
    }
    __syncthreads();
    // the workgroup's pivot, found by every wavefront from the nw candidates
    const double wb = lane < nw ? sbest[buf][lane] : -2.0;
    const int wr = lane < nw ? srow[buf][lane] : INT_MAX;
    const double gb = wave_max_nonneg(fmax(wb, 0.0));
    int gr = wave_min(wb == gb ? wr : INT_MAX);
    if (gr == INT_MAX) gr = wave_min(wb == -1.0 ? wr : INT_MAX);  // NaNs only
    double f[kGjRows];
#pragma unroll
    for (int g = 0; g < kGjRows; ++g) {
      f[g] = -a[g][0];
      if (row[g] == gr) {  // one thread: its row becomes 0 + 1 * prow
        const double d = 1.0 / a[g][0];
        prow[buf][0] = d;
#pragma unroll
        for (int c = 1; c < kPanel; ++c) {
          prow[buf][c] = a[g][c] * d;
          a[g][c] = 0.0;
        }
        f[g] = 1.0;
        free_row[g] = false;
        taken[gr] = k0 + 1;
        piv[k0 + t] = gr;
        if (a[g][0] == 0.0) atomicCAS(flag, 0, k0 + t + 1);  // a NaN is no zero
      }
    }
    __syncthreads();
    // lane c of each wavefront reads entry c of the pivot row and hands it round
    // through scalar registers (reading all 32 entries in every wavefront would
    // wait on LDS)
    const double pr = prow[buf][lane & (kPanel - 1)];
#pragma unroll
    for (int c = 1; c < kPanel; ++c) {
      const double p = lane_read(pr, c);
#pragma unroll
      for (int g = 0; g < kGjRows; ++g) a[g][c - 1] = __builtin_fma(f[g], p, a[g][c]);
    }
    const double p0 = lane_read(pr, 0);
#pragma unroll
    for (int g = 0; g < kGjRows; ++g) a[g][kPanel - 1] = f[g] * p0;
  }
#pragma unroll
  for (int g = 0; g < kGjRows; ++g)
    if (row[g] < m) {
#pragma unroll
      for (int c = 0; c < kPanel; ++c) W[(int64_t)((c + w) % kPanel) * m + row[g]] = a[g][c];
    }
}

// B = A transformed by the panel: row i, column x outside it,
// (i has a pivot of this panel ? 0 : a_ix) + sum_t W(t, i) a(p_t, x); inside it W
__global__ __launch_bounds__(256) void k_gj_update(int m, int k0, int w,
                                                   const double* __restrict__ A,
                                                   const double* __restrict__ W,
                                                   const int32_t* __restrict__ piv,
                                                   const int32_t* __restrict__ taken,
                                                   double* __restrict__ B) {
  __shared__ double ws[kPanel][kTileRows];
  __shared__ double rs[kPanel][kTileCols];
  const int t = threadIdx.x;
  const int r0 = blockIdx.y * kTileRows, x0 = blockIdx.x * kTileCols;
  for (int e = t; e < kTileRows * kPanel; e += 256) {
    const int c = e / kTileRows, r = e % kTileRows;
    ws[c][r] = (r0 + r < m && c < w) ? W[(int64_t)c * m + r0 + r] : 0.0;
  }
  for (int e = t; e < kTileCols * kPanel; e += 256) {
    const int c = e / kTileCols, x = e % kTileCols;
    rs[c][x] = (x0 + x < m && c < w) ? A[(int64_t)piv[k0 + c] * m + x0 + x] : 0.0;
  }
  const int tx = t % 16, ty = t / 16;  // columns tx + 16 q, rows ty + 16 p
  double acc[2][4];
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const int r = r0 + ty + 16 * p;
    const bool keep = r < m && taken[r] != k0 + 1;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int x = x0 + tx + 16 * q;
      acc[p][q] = (keep && x < m) ? A[(int64_t)r * m + x] : 0.0;
    }
  }
  __syncthreads();
#pragma unroll 8
  for (int c = 0; c < kPanel; ++c) {
    double wv[2], rv[4];
#pragma unroll
    for (int p = 0; p < 2; ++p) wv[p] = ws[c][ty + 16 * p];
#pragma unroll
    for (int q = 0; q < 4; ++q) rv[q] = rs[c][tx + 16 * q];
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int q = 0; q < 4; ++q) acc[p][q] = __builtin_fma(wv[p], rv[q], acc[p][q]);
  }
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const int r = r0 + ty + 16 * p;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int x = x0 + tx + 16 * q;
      if (r < m && x < m)
        B[(int64_t)r * m + x] =
            (x >= k0 && x < k0 + w) ? W[(int64_t)(x - k0) * m + r] : acc[p][q];
    }
  }
}

// inv(j, p_i) = A(p_j, i)
__global__ __launch_bounds__(kBlock) void k_gj_unpermute(int m, const double* __restrict__ A,
                                                         const int32_t* __restrict__ piv,
                                                         double* __restrict__ inv) {
  const int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (e >= (int64_t)m * m) return;
  const int j = (int)(e / m), i = (int)(e % m);
  inv[(int64_t)j * m + piv[i]] = A[(int64_t)piv[j] * m + i];
}

// The workspace of one inversion, kept with the context (at most 2 * 1024^2
// doubles): two matrices, the panel, pivot rows, taken flags, the error flag.
int gj_workspace(gh_ctx* ctx, int64_t m, double** a, double** b, double** w, int32_t** piv) {
  const size_t need = sizeof(double) * (2 * m * m + kPanel * m) + sizeof(int32_t) * (2 * m + 2);
  if (ctx->direct_bytes < need) {
    if (ctx->direct_ws) {
      GH_HIP(hipStreamSynchronize(ctx->stream));
      (void)hipFree(ctx->direct_ws);
    }
    ctx->direct_ws = nullptr;
    ctx->direct_bytes = 0;
    if (hipMalloc(&ctx->direct_ws, need) != hipSuccess)
      return fail(GH_ENOMEM, "direct coarse level: allocation failed");
    ctx->direct_bytes = need;
  }
  *a = (double*)ctx->direct_ws;
  *b = *a + m * m;
  *w = *b + m * m;
  *piv = (int32_t*)(*w + kPanel * m);
  return GH_OK;
}

// zeros for the matrix, the taken flags and the error flag
__global__ __launch_bounds__(kBlock) void k_gj_clear(int64_t mm, double* __restrict__ a, int m1,
                                                     int32_t* __restrict__ taken) {
  const int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (e < mm) a[e] = 0.0;
  if (e < m1) taken[e] = 0;
}

int gj_inverse(gh_ctx* ctx, const gh_csr* A, int64_t m, double* inv) {
  double *a, *b, *w;
  int32_t* piv;
  GH_TRY(gj_workspace(ctx, m, &a, &b, &w, &piv));
  int32_t* taken = piv + m;
  int* flag = (int*)(taken + m);
  hipLaunchKernelGGL(k_gj_clear, dim3(grid_for(std::max(m * m, m + 1))), dim3(kBlock), 0,
                     ctx->stream, m * m, a, (int)m + 1, taken);
  hipLaunchKernelGGL(k_scatter_dense, dim3(grid_for(A->n, kBlock / 64)), dim3(kBlock), 0,
                     ctx->stream, A->n, A->ncomp, m, A->rowptr, A->col, (const double*)A->val, a);
  const unsigned threads =
      (unsigned)std::min<int64_t>(kGjThreads, (m + 64 * kGjRows - 1) / (64 * kGjRows) * 64);
  const dim3 tiles((unsigned)((m + kTileCols - 1) / kTileCols),
                   (unsigned)((m + kTileRows - 1) / kTileRows));
  for (int k0 = 0; k0 < m; k0 += kPanel) {
    const int wd = (int)std::min<int64_t>(kPanel, m - k0);
    hipLaunchKernelGGL(k_gj_panel, dim3(1), dim3(threads), 0, ctx->stream, (int)m, k0, wd, a, w, piv,
                       taken, flag);
    hipLaunchKernelGGL(k_gj_update, tiles, dim3(256), 0, ctx->stream, (int)m, k0, wd, a, w, piv,
                       taken, b);
    std::swap(a, b);
  }
  hipLaunchKernelGGL(k_gj_unpermute, dim3(grid_for(m * m)), dim3(kBlock), 0, ctx->stream, (int)m,
                     a, piv, inv);
  GH_HIP(hipGetLastError());
  int hflag = 0;
  GH_HIP(hipMemcpyAsync(&hflag, flag, sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
  GH_HIP(hipStreamSynchronize(ctx->stream));
  if (hflag) return fail(GH_ESINGULAR, "direct coarse level: singular matrix (pivot %d)", hflag);
  return GH_OK;
}

}  // namespace

namespace gh {

void direct_ctx_free(gh_ctx* ctx) {
  if (ctx && ctx->blas) {
    (void)rocblas_destroy_handle((rocblas_handle)ctx->blas);
    ctx->blas = nullptr;
  }
  if (ctx && ctx->direct_ws) {
    (void)hipFree(ctx->direct_ws);
    ctx->direct_ws = nullptr;
    ctx->direct_bytes = 0;
  }
}

int dense_inverse_device(gh_ctx* ctx, const gh_csr* A, double* inv) {
  if (A->prec != GH_F64 || !A->val || !A->rowptr)
    return fail(GH_EINVAL, "direct coarse level: needs the FP64 device matrix");
  const int B = A->ncomp;
  const int64_t m = A->n * B;
  if (m == 0) return GH_OK;
  if (m > 46340) return fail(GH_EINVAL, "direct coarse level: %lld unknowns is too many for a "
                                        "dense inverse", (long long)m);
  // Scalar levels only.  The coarsest Stokes-LPS levels of a channel (27 to 81 nodes,
  // one layer of patches) are singular to rounding (condition 2e16 to 1e17): what
  // their inverse holds is rounding of the elimination, so they keep the one whose
  // results their solvers have had so far.  Nothing is lost on the solve: both
  // inverses are applied by the same kernel.
  if (B == 1 && m <= kGjMax) return gj_inverse(ctx, A, m, inv);
  if (!ctx->blas) {
    rocblas_handle h = nullptr;
    if (rocblas_create_handle(&h) != rocblas_status_success)
      return fail(GH_EHIP, "direct coarse level: rocblas_create_handle failed");
    ctx->blas = h;
  }
  rocblas_handle h = (rocblas_handle)ctx->blas;
  if (rocblas_set_stream(h, ctx->stream) != rocblas_status_success)
    return fail(GH_EHIP, "direct coarse level: rocblas_set_stream failed");
  rocblas_int* ipiv = nullptr;
  rocblas_int* info = nullptr;
  if (hipMalloc((void**)&ipiv, sizeof(rocblas_int) * m) != hipSuccess ||
      hipMalloc((void**)&info, sizeof(rocblas_int) * 2) != hipSuccess) {
    if (ipiv) (void)hipFree(ipiv);
    return fail(GH_ENOMEM, "direct coarse level: allocation failed");
  }
  int rc = GH_OK;
  // the row-major scatter is A^T in column-major order; the column-major
  // inverse of A^T read row-major is A^-1
  hipLaunchKernelGGL(k_fill0<double>, dim3((unsigned)std::min<int64_t>((m * m + kBlock - 1) / kBlock, 8192)),
                     dim3(kBlock), 0, ctx->stream, m * m, inv);
  hipLaunchKernelGGL(k_scatter_dense, dim3(grid_for(A->n, kBlock / 64)), dim3(kBlock), 0,
                     ctx->stream, A->n, B, m, A->rowptr, A->col, (const double*)A->val, inv);
  if (hipGetLastError() != hipSuccess) rc = fail(GH_EHIP, "direct coarse level: scatter");
  if (!rc && rocsolver_dgetrf(h, (rocblas_int)m, (rocblas_int)m, inv, (rocblas_int)m, ipiv,
                              info) != rocblas_status_success)
    rc = fail(GH_EHIP, "direct coarse level: rocsolver_dgetrf failed");
  if (!rc && rocsolver_dgetri(h, (rocblas_int)m, inv, (rocblas_int)m, ipiv, info + 1) !=
                 rocblas_status_success)
    rc = fail(GH_EHIP, "direct coarse level: rocsolver_dgetri failed");
  rocblas_int hinfo[2] = {0, 0};
  if (!rc && hipMemcpyAsync(hinfo, info, sizeof(hinfo), hipMemcpyDeviceToHost, ctx->stream) !=
                 hipSuccess)
    rc = fail(GH_EHIP, "direct coarse level: info copy");
  if (!rc && hipStreamSynchronize(ctx->stream) != hipSuccess)
    rc = fail(GH_EHIP, "direct coarse level: sync");
  if (!rc && (hinfo[0] != 0 || hinfo[1] != 0))
    rc = fail(GH_ESINGULAR, "direct coarse level: singular matrix (pivot %d)", (int)hinfo[0]);
  (void)hipFree(ipiv);
  (void)hipFree(info);
  return rc;
}

}  // namespace gh
