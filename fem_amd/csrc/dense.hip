// dense.hip -- dense inverse of each cell's coarsest operator (n = 3 V_c <= 648
// unknowns), formed on the device.
//
// The operator A + (d / V) Z Z^T (Z the three constant fields, d the mean
// diagonal) is symmetric positive definite, so it is inverted in place by the
// symmetric sweep (Gauss-Jordan without pivoting): sweeping pivot block K of a
// symmetric matrix replaces A_KK by -P, P = A_KK^-1, A_iK by A_iK P and every
// other A_ij by A_ij - A_iK P A_Kj, and the matrix stays symmetric; after all
// blocks it is -A^-1.  All arithmetic is FP64.
//
// The work is tiny for the device (n^3 multiply-adds: 53 M for the 375
// unknowns of a 40^3 cell), so what bounds it is the chain of n pivots.  Up to
// kSmallDense unknowns the matrix lives in one workgroup's LDS and a pivot
// costs two barriers; above, kPanel pivots share a pair of launches (panel,
// then update of all tiles).  On one host core the same inverse (Cholesky and
// n pairs of triangular solves) took 22 ms per cell of 375 unknowns, nine
// tenths of a 40^3 cell's whole solve: eight 40^3 cells with their tensors went
// from 204 to 30 ms, an uneven batch of 64 cells (13 of them 40^3) from 457 to
// 372 ms.
#include <hip/hip_runtime.h>

#include <stdexcept>

#include "device_common.hpp"
#include "kernels.hpp"

namespace femh {

constexpr int kSmallDense = 88;  // matrix of 88 x 88 doubles: 62 KB of LDS
constexpr int kPanel = 32;       // pivots per panel
constexpr int kUpd = 64;         // tile edge of the update

// A[s] (row-major, unknown c V + N) from the 27-point stencils: a thread adds
// up the blocks that couple node N to node M (several on a level with a
// dimension of 2, where offsets wrap onto each other)
template <typename T>
__global__ __launch_bounds__(kBlock) void k_dense_assemble(Dims g, const T *__restrict__ S, double *__restrict__ A) {
  const int smp = blockIdx.y, V = g.V, n = 3 * V;
  const T *__restrict__ Ss = S + (size_t)smp * 243 * V;
  double d = 0;
  for (int t = threadIdx.x; t < n; t += kBlock) d += (double)Ss[stencil_index(13, 4 * (t / V), V, t % V)];
  const double shift = block_sum(d) / n / V;
  const int t = blockIdx.x * kBlock + threadIdx.x;
  if (t >= V * V) return;
  const int N = t / V, M = t - N * V;
  int i, j, k;
  node_ijk(g, N, i, j, k);
  double a[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  for (int o = 0; o < 27; o++) {
    const int ni = (i + o / 9 - 1 + g.nx) % g.nx, nj = (j + (o / 3) % 3 - 1 + g.ny) % g.ny,
              nk = (k + o % 3 - 1 + g.nz) % g.nz;
    if ((ni * g.ny + nj) * g.nz + nk != M) continue;
#pragma unroll
    for (int q = 0; q < 9; q++) a[q] += (double)Ss[stencil_index(o, q, V, N)];
  }
  double *__restrict__ As = A + (size_t)smp * n * n;
#pragma unroll
  for (int c = 0; c < 3; c++)
#pragma unroll
    for (int e = 0; e < 3; e++)
      As[(size_t)(c * V + N) * n + e * V + M] = a[3 * c + e] + (c == e ? shift : 0.0);
}

// one workgroup per cell, the matrix in LDS: thread (ty, tx) of 32 x 32 owns
// the entries (ty + 32 a, tx + 32 b)
template <typename T>
__global__ __launch_bounds__(1024) void k_dense_small(int n, const double *__restrict__ A, T *__restrict__ out,
                                                      int *__restrict__ bad) {
  __shared__ double m[kSmallDense * kSmallDense];
  const int smp = blockIdx.x, tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  constexpr int Q = (kSmallDense + 31) / 32;
  const double *__restrict__ As = A + (size_t)smp * n * n;
  for (int t = threadIdx.x; t < n * n; t += 1024) m[t] = As[t];
  __syncthreads();
  bool ok = true;
  for (int k = 0; k < n; k++) {
    const double d = m[k * n + k];
    ok = ok && d > 0;
    const double di = 1.0 / d;
    double v[Q][Q];
#pragma unroll
    for (int a = 0; a < Q; a++)
#pragma unroll
      for (int b = 0; b < Q; b++) {
        const int i = ty + 32 * a, j = tx + 32 * b;
        if (i >= n || j >= n) continue;
        const double rk = m[k * n + j] * di;
        v[a][b] = i == k ? (j == k ? -di : rk) : (j == k ? m[i * n + k] * di : m[i * n + j] - m[i * n + k] * rk);
      }
    __syncthreads();
#pragma unroll
    for (int a = 0; a < Q; a++)
#pragma unroll
      for (int b = 0; b < Q; b++) {
        const int i = ty + 32 * a, j = tx + 32 * b;
        if (i < n && j < n) m[i * n + j] = v[a][b];
      }
    __syncthreads();
  }
  T *__restrict__ os = out + (size_t)smp * n * n;
  for (int t = threadIdx.x; t < n * n; t += 1024) os[t] = (T)(-m[t]);
  if (threadIdx.x == 0) bad[smp] = ok ? 0 : 1;
}

// Pivot block k0 .. k0 + kb - 1: every workgroup sweeps the block in LDS and
// forms 64 columns of the panel, old rows A_K,: and new rows P A_K,: (-P in
// the pivot columns) into pan[s][2][kPanel][n]
__global__ __launch_bounds__(kBlock) void k_dense_panel(int n, int k0, int kb, const double *__restrict__ A,
                                                        double *__restrict__ pan, int *__restrict__ bad) {
  __shared__ double P[kPanel][kPanel + 1], Qs[kPanel][kUpd];
  const int smp = blockIdx.y, j0 = blockIdx.x * kUpd, tid = threadIdx.x;
  const double *__restrict__ As = A + (size_t)smp * n * n;
  for (int t = tid; t < kPanel * kPanel; t += kBlock) {
    const int r = t / kPanel, c = t % kPanel;
    P[r][c] = (r < kb && c < kb) ? As[(size_t)(k0 + r) * n + k0 + c] : 0.0;
  }
  for (int t = tid; t < kPanel * kUpd; t += kBlock) {
    const int r = t / kUpd, c = t % kUpd;
    Qs[r][c] = (r < kb && j0 + c < n) ? As[(size_t)(k0 + r) * n + j0 + c] : 0.0;
  }
  __syncthreads();
  const int tx = tid & 31, ty = tid >> 5;  // entries (ty + 8 a, tx)
  bool ok = true;
  for (int k = 0; k < kb; k++) {
    const double d = P[k][k];
    ok = ok && d > 0;
    const double di = 1.0 / d, rk = P[k][tx] * di;
    double v[4];
#pragma unroll
    for (int a = 0; a < 4; a++) {
      const int i = ty + 8 * a;
      v[a] = i == k ? (tx == k ? -di : rk) : (tx == k ? P[i][k] * di : P[i][tx] - P[i][k] * rk);
    }
    __syncthreads();
#pragma unroll
    for (int a = 0; a < 4; a++)
      if (ty + 8 * a < kb && tx < kb) P[ty + 8 * a][tx] = v[a];
    __syncthreads();
  }
  if (blockIdx.x == 0 && tid == 0 && !ok) bad[smp] = 1;
  double *__restrict__ old = pan + (size_t)smp * 2 * kPanel * n, *__restrict__ neu = old + (size_t)kPanel * n;
  const int c = tid & 63, r0 = (tid >> 6) * 8, j = j0 + c;
  if (j >= n) return;
  double acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  for (int q = 0; q < kb; q++) {
    const double u = Qs[q][c];
#pragma unroll
    for (int a = 0; a < 8; a++) acc[a] -= P[r0 + a][q] * u;
  }
  const bool piv = j >= k0 && j < k0 + kb;
#pragma unroll
  for (int a = 0; a < 8; a++) {
    const int r = r0 + a;
    old[(size_t)r * n + j] = Qs[r][c];
    neu[(size_t)r * n + j] = r < kb ? (piv ? P[r][j - k0] : acc[a]) : 0.0;
  }
}

// all tiles of one sweep: A_ij -= A_iK (P A_K,:)_j, the pivot rows and columns
// from the panel; after the last block (out given) -A goes to out
template <typename T>
__global__ __launch_bounds__(kBlock) void k_dense_update(int n, int k0, int kb, double *__restrict__ A,
                                                         const double *__restrict__ pan, T *__restrict__ out) {
  __shared__ double O[kPanel][kUpd], W[kPanel][kUpd];
  const int smp = blockIdx.z, i0 = blockIdx.y * kUpd, j0 = blockIdx.x * kUpd, tid = threadIdx.x;
  const double *__restrict__ old = pan + (size_t)smp * 2 * kPanel * n, *__restrict__ neu = old + (size_t)kPanel * n;
  for (int t = tid; t < kPanel * kUpd; t += kBlock) {
    const int r = t / kUpd, c = t % kUpd;
    O[r][c] = i0 + c < n ? old[(size_t)r * n + i0 + c] : 0.0;
    W[r][c] = j0 + c < n ? neu[(size_t)r * n + j0 + c] : 0.0;
  }
  __syncthreads();
  const int tx = tid & 15, ty = tid >> 4;  // entries (ty + 16 a, tx + 16 b)
  double acc[4][4] = {};
#pragma unroll 4
  for (int r = 0; r < kPanel; r++) {
    double o[4], w[4];
#pragma unroll
    for (int a = 0; a < 4; a++) {
      o[a] = O[r][ty + 16 * a];
      w[a] = W[r][tx + 16 * a];
    }
#pragma unroll
    for (int a = 0; a < 4; a++)
#pragma unroll
      for (int b = 0; b < 4; b++) acc[a][b] += o[a] * w[b];
  }
  double *__restrict__ As = A + (size_t)smp * n * n;
  T *__restrict__ os = out ? out + (size_t)smp * n * n : nullptr;
#pragma unroll
  for (int a = 0; a < 4; a++)
#pragma unroll
    for (int b = 0; b < 4; b++) {
      const int i = i0 + ty + 16 * a, j = j0 + tx + 16 * b;
      if (i >= n || j >= n) continue;
      const size_t e = (size_t)i * n + j;
      double v;
      if (i >= k0 && i < k0 + kb)
        v = W[i - k0][tx + 16 * b];
      else if (j >= k0 && j < k0 + kb)
        v = neu[(size_t)(j - k0) * n + i];
      else
        v = As[e] - acc[a][b];
      if (os)
        os[e] = (T)(-v);
      else
        As[e] = v;
    }
}

size_t dense_work_doubles(int n, int B) { return ((size_t)n * n + (n > kSmallDense ? 2 * (size_t)kPanel * n : 0)) * B; }

template <typename T>
void launch_dense_inverse(const Dims &g, int nb, const T *S, double *work, T *Ainv, int *bad, hipStream_t s) {
  const int n = 3 * g.V;
  launch_fill<int>(nb, bad, 0, s);
  hipLaunchKernelGGL(k_dense_assemble<T>, dim3((g.V * g.V + kBlock - 1) / kBlock, nb), dim3(kBlock), 0, s, g, S, work);
  if (n <= kSmallDense) {
    hipLaunchKernelGGL(k_dense_small<T>, dim3(nb), dim3(1024), 0, s, n, work, Ainv, bad);
    return;
  }
  double *pan = work + (size_t)n * n * nb;
  const int tiles = (n + kUpd - 1) / kUpd;
  for (int k0 = 0; k0 < n; k0 += kPanel) {
    const int kb = n - k0 < kPanel ? n - k0 : kPanel;
    hipLaunchKernelGGL(k_dense_panel, dim3(tiles, nb), dim3(kBlock), 0, s, n, k0, kb, work, pan, bad);
    hipLaunchKernelGGL(k_dense_update<T>, dim3(tiles, tiles, nb), dim3(kBlock), 0, s, n, k0, kb, work, pan,
                       k0 + kb >= n ? Ainv : nullptr);
  }
}

template void launch_dense_inverse<double>(const Dims &, int, const double *, double *, double *, int *, hipStream_t);
template void launch_dense_inverse<float>(const Dims &, int, const float *, double *, float *, int *, hipStream_t);

}  // namespace femh
