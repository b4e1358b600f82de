// dense.hip -- dense inverse of each cell's coarsest operator (n = 3 V_c <= 648
// unknowns), formed on the device in FP64.
//
// The operator A + (d / V) Z Z^T (Z the three constant fields, d the mean
// diagonal) is symmetric positive definite: Cholesky A = L L^T, then a forward
// and a backward substitution for every unit column.  Every entry is formed
// by the same operations in the same order as the plain sequential algorithm
// (ascending index in each sum, product and difference rounded apart: no
// fused multiply-add), so the inverse does not depend on the split: the FP32
// multigrid that uses it gives the same bits as with a host factorisation.
//
// What bounds it is the chain of dependent operations, not their number (n^3
// multiply-adds: 53 M for the 375 unknowns of a 40^3 cell).  The factor goes
// by panels of kPanel columns, two launches each (panel, trailing update);
// the forward substitution by blocks of kPanel rows within one workgroup; the
// backward substitution sums in ascending order from the unknown found last,
// which is one chain of n^2 / 2 terms per column: a column per lane, the
// columns found so far in LDS.  Eight cells of 375 unknowns: panels and updates
// 0.3 ms, forward 0.48 ms, backward 0.62 ms.  On one host core the same took 22
// ms per cell, nine tenths of a 40^3 cell's whole solve (eight such cells with
// their tensors: 203 ms then, 30.0 ms now; an uneven batch of 64 cells, 13 of
// them 40^3: 495 and 268 ms).
#include <hip/hip_runtime.h>

#include <stdexcept>

#include "device_common.hpp"
#include "kernels.hpp"

namespace femh {

constexpr int kDenseMax = 648;
constexpr int kPanel = 32;  // columns per panel
constexpr int kUpd = 64;    // tile edge of the trailing update, columns per forward workgroup
constexpr int kFwd = 512;        // threads of a forward workgroup
constexpr int kSmallDense = 88;  // matrix and inverse in LDS: 121 KB

// the mean diagonal over V, summed in index order by one thread (dg: n values
// of LDS); all threads of the block call and receive it
template <typename T>
__device__ __forceinline__ double dense_shift(const T *__restrict__ Ss, int V, double *dg, double *sh) {
  const int n = 3 * V;
  for (int t = threadIdx.x; t < n; t += blockDim.x) dg[t] = (double)Ss[stencil_index(13, 4 * (t / V), V, t % V)];
  __syncthreads();
  if (threadIdx.x == 0) {
    double d = 0;
    for (int t = 0; t < n; t++) d += dg[t];
    *sh = d / n / V;
  }
  __syncthreads();
  return *sh;
}

// the 3x3 block of nodes N, M: the sum of the stencil blocks that couple N to M
// (several on a level with a dimension of 2, where offsets wrap onto each other)
template <typename T>
__device__ __forceinline__ void dense_block(const Dims &g, const T *__restrict__ Ss, int N, int M, double (&a)[9]) {
  int i, j, k;
  node_ijk(g, N, i, j, k);
#pragma unroll
  for (int q = 0; q < 9; q++) a[q] = 0;
  for (int o = 0; o < 27; o++) {
    const int ni = (i + o / 9 - 1 + g.nx) % g.nx, nj = (j + (o / 3) % 3 - 1 + g.ny) % g.ny,
              nk = (k + o % 3 - 1 + g.nz) % g.nz;
    if ((ni * g.ny + nj) * g.nz + nk != M) continue;
#pragma unroll
    for (int q = 0; q < 9; q++) a[q] += (double)Ss[stencil_index(o, q, g.V, N)];
  }
}

// A[s] (row-major, unknown c V + N) from the 27-point stencils, a thread per
// node pair
template <typename T>
__global__ __launch_bounds__(kBlock) void k_dense_assemble(Dims g, const T *__restrict__ S, double *__restrict__ A) {
  const int smp = blockIdx.y, V = g.V, n = 3 * V;
  const T *__restrict__ Ss = S + (size_t)smp * 243 * V;
  __shared__ double dg[kDenseMax], sh;
  const double shift = dense_shift(Ss, V, dg, &sh);
  const int t = blockIdx.x * kBlock + threadIdx.x;
  if (t >= V * V) return;
  const int N = t / V, M = t - N * V;
  double a[9];
  dense_block(g, Ss, N, M, a);
  double *__restrict__ As = A + (size_t)smp * n * n;
#pragma unroll
  for (int c = 0; c < 3; c++)
#pragma unroll
    for (int e = 0; e < 3; e++)
      As[(size_t)(c * V + N) * n + e * V + M] = a[3 * c + e] + (c == e ? shift : 0.0);
}

// Up to kSmallDense unknowns: one workgroup per cell does it all in LDS, factor
// by columns (three barriers each), then a column of the inverse per thread.
// (n = 24, the coarsest level of 16^3, 32^3, 64^3 cells: one launch of 52 us; by
// the panel kernels it was seven launches and 50 us more for the call.)
template <typename T>
__global__ __launch_bounds__(kBlock) void k_dense_small(Dims g, const T *__restrict__ S, T *__restrict__ out,
                                                        int *__restrict__ bad) {
#pragma clang fp contract(off)
  __shared__ double m[kSmallDense * kSmallDense], x[kSmallDense * kSmallDense], dg[kSmallDense], sh;
  const int smp = blockIdx.x, V = g.V, n = 3 * V, tid = threadIdx.x;
  const T *__restrict__ Ss = S + (size_t)smp * 243 * V;
  const double shift = dense_shift(Ss, V, dg, &sh);
  for (int t = tid; t < V * V; t += kBlock) {
    const int N = t / V, M = t - N * V;
    double a[9];
    dense_block(g, Ss, N, M, a);
#pragma unroll
    for (int c = 0; c < 3; c++)
#pragma unroll
      for (int e = 0; e < 3; e++) m[(c * V + N) * n + e * V + M] = a[3 * c + e] + (c == e ? shift : 0.0);
  }
  __syncthreads();
  const int tx = tid & 15, ty = tid >> 4;
  bool ok = true;
  for (int j = 0; j < n; j++) {
    const double p = m[j * n + j];
    ok = ok && p > 0;
    const double d = sqrt(p);
    __syncthreads();
    for (int i = j + tid; i < n; i += kBlock) m[i * n + j] = i == j ? d : m[i * n + j] / d;
    __syncthreads();
    for (int i = j + 1 + ty; i < n; i += 16)
      for (int c = j + 1 + tx; c <= i; c += 16) m[i * n + c] = m[i * n + c] - m[i * n + j] * m[c * n + j];
    __syncthreads();
  }
  if (tid == 0) bad[smp] = ok ? 0 : 1;
  T *__restrict__ os = out + (size_t)smp * n * n;
  const int c = tid;
  if (c >= n) return;
  for (int i = 0; i < n; i++) {
    double s = i == c ? 1.0 : 0.0;
    if (i >= c) {
#pragma unroll 8
      for (int k = c; k < i; k++) s = s - m[i * n + k] * x[k * n + c];
      s = s / m[i * n + i];
    }
    x[i * n + c] = s;
  }
  for (int i = n - 1; i >= 0; i--) {
    double s = x[i * n + c];
#pragma unroll 8
    for (int k = i + 1; k < n; k++) s = s - m[k * n + i] * x[k * n + c];
    s = s / m[i * n + i];
    x[i * n + c] = s;
    os[i * n + c] = (T)s;
  }
}

// Panel k0 .. k0 + kb - 1 of the factor: every workgroup factors the diagonal
// block in LDS and finishes 64 rows below it, one thread per row (its kPanel
// entries in registers).  L goes to Lf and, transposed, to Lt; A keeps the
// trailing matrix only (other workgroups still read the block).
__global__ __launch_bounds__(kBlock) void k_chol_panel(int n, int k0, int kb, const double *__restrict__ A,
                                                       double *__restrict__ Lf, double *__restrict__ Lt,
                                                       int *__restrict__ bad) {
#pragma clang fp contract(off)
  __shared__ double D[kPanel][kPanel + 1];
  const int smp = blockIdx.y, tid = threadIdx.x;
  const size_t ms = (size_t)smp * n * n;
  const double *__restrict__ As = A + ms;
  for (int t = tid; t < kPanel * kPanel; t += kBlock) {
    const int r = t / kPanel, c = t % kPanel;
    D[r][c] = (r < kb && c < kb) ? As[(size_t)(k0 + r) * n + k0 + c] : (r == c ? 1.0 : 0.0);
  }
  __syncthreads();
  const int tx = tid & 31, ty = tid >> 5;
  bool ok = true;
  for (int j = 0; j < kb; j++) {
    const double p = D[j][j];
    ok = ok && p > 0;
    const double d = sqrt(p);
    __syncthreads();
    if (tid == 0) D[j][j] = d;
    if (tid > j && tid < kPanel) D[tid][j] = D[tid][j] / d;
    __syncthreads();
#pragma unroll
    for (int a = 0; a < 4; a++) {
      const int i = ty + 8 * a;
      if (tx > j && i >= tx) D[i][tx] = D[i][tx] - D[i][j] * D[tx][j];
    }
    __syncthreads();
  }
  double *__restrict__ Ls = Lf + ms, *__restrict__ Ts = Lt + ms;
  if (blockIdx.x == 0) {
    if (tid == 0 && !ok) bad[smp] = 1;
    for (int t = tid; t < kPanel * kPanel; t += kBlock) {
      const int r = t / kPanel, c = t % kPanel;
      if (r >= kb || c > r) continue;
      Ls[(size_t)(k0 + r) * n + k0 + c] = D[r][c];
      Ts[(size_t)(k0 + c) * n + k0 + r] = D[r][c];
    }
  }
  // (rows below exist only under a full block, kb = kPanel)
  const int i = k0 + kPanel + blockIdx.x * kUpd + tid;
  if (tid >= kUpd || i >= n) return;
  double l[kPanel];
#pragma unroll
  for (int j = 0; j < kPanel; j++) l[j] = As[(size_t)i * n + k0 + j];
#pragma unroll
  for (int j = 0; j < kPanel; j++) {
    l[j] = l[j] / D[j][j];
#pragma unroll
    for (int m = j + 1; m < kPanel; m++) l[m] = l[m] - l[j] * D[m][j];
  }
#pragma unroll
  for (int j = 0; j < kPanel; j++) {
    Ls[(size_t)i * n + k0 + j] = l[j];
    Ts[(size_t)(k0 + j) * n + i] = l[j];
  }
}

// trailing update of a full panel: A_ij -= sum_m L_im L_jm, m ascending, for
// the tiles on and below the diagonal of the rows from k1 = k0 + kPanel on
__global__ __launch_bounds__(kBlock) void k_chol_update(int n, int k0, double *__restrict__ A,
                                                        const double *__restrict__ Lf) {
#pragma clang fp contract(off)
  if (blockIdx.x > blockIdx.y) return;
  __shared__ double Li[kUpd][kPanel + 1], Lj[kUpd][kPanel + 1];
  const int smp = blockIdx.z, tid = threadIdx.x, k1 = k0 + kPanel;
  const int i0 = k1 + blockIdx.y * kUpd, j0 = k1 + blockIdx.x * kUpd;
  const size_t ms = (size_t)smp * n * n;
  const double *__restrict__ Ls = Lf + ms;
  for (int t = tid; t < kUpd * kPanel; t += kBlock) {
    const int r = t / kPanel, c = t % kPanel;
    Li[r][c] = i0 + r < n ? Ls[(size_t)(i0 + r) * n + k0 + c] : 0.0;
    Lj[r][c] = j0 + r < n ? Ls[(size_t)(j0 + r) * n + k0 + c] : 0.0;
  }
  const int tx = tid & 15, ty = tid >> 4;  // entries (ty + 16 a, tx + 16 b)
  double *__restrict__ As = A + ms;
  double v[4][4];
#pragma unroll
  for (int a = 0; a < 4; a++)
#pragma unroll
    for (int b = 0; b < 4; b++) {
      const int i = i0 + ty + 16 * a, j = j0 + tx + 16 * b;
      v[a][b] = (i < n && j < n) ? As[(size_t)i * n + j] : 0.0;
    }
  __syncthreads();
#pragma unroll 4
  for (int m = 0; m < kPanel; m++) {
    double x[4], y[4];
#pragma unroll
    for (int a = 0; a < 4; a++) {
      x[a] = Li[ty + 16 * a][m];
      y[a] = Lj[tx + 16 * a][m];
    }
#pragma unroll
    for (int a = 0; a < 4; a++)
#pragma unroll
      for (int b = 0; b < 4; b++) v[a][b] = v[a][b] - x[a] * y[b];
  }
#pragma unroll
  for (int a = 0; a < 4; a++)
#pragma unroll
    for (int b = 0; b < 4; b++) {
      const int i = i0 + ty + 16 * a, j = j0 + tx + 16 * b;
      if (i < n && j < n) As[(size_t)i * n + j] = v[a][b];
    }
}

// forward substitution L y = e_c for 64 columns c of a cell, a column per lane:
// per block of kPanel rows, wave 0 solves the block in LDS and all 8 waves then update the rows below, two rows
// at a time per wave, with the block's solution in registers.  Rows above the
// first block that holds one of the columns stay unwritten (they are zero).
__global__ __launch_bounds__(kFwd) void k_chol_forward(int n, const double *__restrict__ Lf, double *__restrict__ Y) {
#pragma clang fp contract(off)
  __shared__ double yb[kPanel][kUpd], D[kPanel][kPanel + 1];
  const int smp = blockIdx.y, lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = blockIdx.x * kUpd + lane;
  const bool live = c < n;
  const int first = blockIdx.x * kUpd;  // (a multiple of kPanel)
  const double *__restrict__ Ls = Lf + (size_t)smp * n * n;
  double *__restrict__ Ys = Y + (size_t)smp * n * n;
  for (int k0 = first; k0 < n; k0 += kPanel) {
    const int kb = min(kPanel, n - k0);
    for (int t = threadIdx.x; t < kPanel * kPanel; t += kFwd) {
      const int r = t / kPanel, q = t % kPanel;
      D[r][q] = (r < kb && q <= r) ? Ls[(size_t)(k0 + r) * n + k0 + q] : (r == q ? 1.0 : 0.0);
    }
    __syncthreads();
    if (w == 0) {
      for (int r = 0; r < kb; r++)
        yb[r][lane] = k0 == first ? (k0 + r == c ? 1.0 : 0.0) : (live ? Ys[(size_t)(k0 + r) * n + c] : 0.0);
      for (int r = 0; r < kb; r++) {
        const double yr = yb[r][lane] / D[r][r];
        yb[r][lane] = yr;
        if (live) Ys[(size_t)(k0 + r) * n + c] = yr;
#pragma unroll 8
        for (int m = r + 1; m < kb; m++) yb[m][lane] = yb[m][lane] - D[m][r] * yr;
      }
    }
    __syncthreads();
    // (rows below exist only under a full block)
    double y[kPanel];
#pragma unroll
    for (int r = 0; r < kPanel; r++) y[r] = yb[r][lane];
    for (int i = k0 + kPanel + w; i < n; i += kFwd / 32) {
      const int i2 = i + kFwd / 64;
      const bool two = i2 < n;
      const double *__restrict__ r1 = Ls + (size_t)i * n + k0, *__restrict__ r2 = two ? Ls + (size_t)i2 * n + k0 : r1;
      double s1, s2;
      if (k0 == first) {
        s1 = i == c ? 1.0 : 0.0;
        s2 = i2 == c ? 1.0 : 0.0;
      } else {
        s1 = live ? Ys[(size_t)i * n + c] : 0.0;
        s2 = live && two ? Ys[(size_t)i2 * n + c] : 0.0;
      }
#pragma unroll
      for (int m = 0; m < kPanel; m++) {
        s1 = s1 - r1[m] * y[m];
        s2 = s2 - r2[m] * y[m];
      }
      if (live) {
        Ys[(size_t)i * n + c] = s1;
        if (two) Ys[(size_t)i2 * n + c] = s2;
      }
    }
    __syncthreads();
  }
}

// backward substitution L^T x = y for NC columns of a cell.  Wave 0 runs the
// chains, a column per lane; the other three waves form the next row's
// products L_ki x_k (k past the row in progress) meanwhile, so a chain step is
// one subtraction of a value read from LDS.  (One wave that
// also formed its products: 1.63 ms for the eight cells of 375 unknowns.)  Rows above a column's forward block: y = 0.
template <typename T, int NMAX, int NC>
__global__ __launch_bounds__(kBlock) void k_chol_backward(int n, const double *__restrict__ Lt,
                                                          const double *__restrict__ Y, T *__restrict__ out) {
#pragma clang fp contract(off)
  constexpr int XS = NC + 1, PS = NMAX + 2, NP = kBlock - 64, Q = (NMAX + NP - 1) / NP;
  __shared__ double x[NMAX * XS], pr[2][NC * PS];
  const int smp = blockIdx.y, tid = threadIdx.x;
  const int c0 = blockIdx.x * NC, first = c0 / kUpd * kUpd;
  const double *__restrict__ Ts = Lt + (size_t)smp * n * n;
  const double *__restrict__ Ys = Y + (size_t)smp * n * n;
  T *__restrict__ os = out + (size_t)smp * n * n;
  if (tid < 64) {
    const int lane = tid, c = c0 + lane;
    const bool live = lane < NC && c < n;
    double y = live ? Ys[(size_t)(n - 1) * n + c] : 0.0, xp = 0.0;
    for (int i = n - 1; i >= 0; i--) {
      if (live) {
        const double *row = Ts + (size_t)i * n;
        double s = y;
        const double d = row[i];
        if (i + 1 < n) s = s - row[i + 1] * xp;
        y = i > first ? Ys[(size_t)(i - 1) * n + c] : 0.0;  // (ahead of the chain)
        const double *p = &pr[i & 1][lane * PS];
#pragma unroll 16
        for (int k = i + 2; k < n; k++) s = s - p[k];
        xp = s / d;
        x[i * XS + lane] = xp;
        os[(size_t)i * n + c] = (T)xp;
      }
      __syncthreads();
    }
    return;
  }
  const int t = tid - 64;
  // products of row i - 1 need x_k for k > i: all found before row i began
  double l[Q];
  auto fetch = [&](int i) {
#pragma unroll
    for (int q = 0; q < Q; q++) {
      const int k = t + q * NP;
      l[q] = (i >= 0 && k > i + 1 && k < n) ? Ts[(size_t)i * n + k] : 0.0;
    }
  };
  fetch(n - 2);
  for (int i = n - 1; i >= 0; i--) {
    // (row i - 1, into the buffer that row i does not read)
    double *p = pr[(i - 1) & 1];
    double lc[Q];
#pragma unroll
    for (int q = 0; q < Q; q++) lc[q] = l[q];
    fetch(i - 2);
#pragma unroll
    for (int q = 0; q < Q; q++) {
      const int k = t + q * NP;
      if (k > i && k < n) {
#pragma unroll
        for (int e = 0; e < NC; e++) p[e * PS + k] = lc[q] * x[k * XS + e];
      }
    }
    __syncthreads();
  }
}

size_t dense_work_doubles(int n, int nb) { return n <= kSmallDense ? 0 : (size_t)3 * n * n * nb; }

template <typename T>
void launch_dense_inverse(const Dims &g, int nb, const T *S, double *work, T *Ainv, int *bad, hipStream_t s) {
  const int n = 3 * g.V;
  if (n > kDenseMax) throw std::runtime_error("coarsest level too large for the dense inverse");
  if (n <= kSmallDense) {
    hipLaunchKernelGGL(k_dense_small<T>, dim3(nb), dim3(kBlock), 0, s, g, S, Ainv, bad);
    return;
  }
  double *A = work, *Lf = A + (size_t)n * n * nb, *Lt = Lf + (size_t)n * n * nb;
  launch_fill<int>(nb, bad, 0, s);
  hipLaunchKernelGGL(k_dense_assemble<T>, dim3((g.V * g.V + kBlock - 1) / kBlock, nb), dim3(kBlock), 0, s, g, S, A);
  for (int k0 = 0; k0 < n; k0 += kPanel) {
    const int kb = n - k0 < kPanel ? n - k0 : kPanel, below = n - k0 - kb, tiles = (below + kUpd - 1) / kUpd;
    hipLaunchKernelGGL(k_chol_panel, dim3(tiles > 0 ? tiles : 1, nb), dim3(kBlock), 0, s, n, k0, kb, A, Lf, Lt, bad);
    if (below > 0)
      hipLaunchKernelGGL(k_chol_update, dim3(tiles, tiles, nb), dim3(kBlock), 0, s, n, k0, A, Lf);
  }
  // (A is used up: the forward results go over it)
  hipLaunchKernelGGL(k_chol_forward, dim3((n + kUpd - 1) / kUpd, nb), dim3(kFwd), 0, s, n, Lf, A);
  // 16 columns per backward workgroup while their products fit the LDS
  if (n <= 384)
    hipLaunchKernelGGL((k_chol_backward<T, 384, 16>), dim3((n + 15) / 16, nb), dim3(kBlock), 0, s, n, Lt, A, Ainv);
  else
    hipLaunchKernelGGL((k_chol_backward<T, kDenseMax, 8>), dim3((n + 7) / 8, nb), dim3(kBlock), 0, s, n, Lt, A, Ainv);
}

template void launch_dense_inverse<double>(const Dims &, int, const double *, double *, double *, int *, hipStream_t);
template void launch_dense_inverse<float>(const Dims &, int, const float *, double *, float *, int *, hipStream_t);

}  // namespace femh
