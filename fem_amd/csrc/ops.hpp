// ops.hpp -- fused operator kernels (ops.hip): K u with a staging transform
// applied to the input and a Chebyshev/PCG epilogue applied to the output,
// so that one smoothing step is one kernel.
//
// Staging (value of the input at every node the stencil touches):
//   ST_PLAIN     u
//   ST_DSCALE    u * theta_inv / D              (first Chebyshev step from x = 0)
//   ST_PROLONG   u + P xc                       (coarse correction added on the fly)
//   ST_DPROLONG  u * theta_inv / D + P xc       (u = b: degree-1 pre-smoothing and
//                                                coarse correction in one)
//   ST_PUPD      u + beta u2                    (PCG direction p = z + beta p_old,
//                                                beta per RHS from a device array)
//   ST_PUPDX     the same, and x += alpha u2 at the owned node: the solution
//                update of the previous iteration, whose direction u2 is
//   ST_RUPD      (u - alpha u2) * theta_inv / D (u = r, u2 = q = A p: the residual
//                update r' = r - alpha q and the degree-1 pre-smoothing; pout = r',
//                and with `dot` the FP64 partial of r'.r'; b is r' itself)
// (D enters as its precomputed inverse: no divisions in the kernels.  beta of
// ST_PUPDX and alpha of ST_RUPD are formed from the partials of the dot products
// by every workgroup: a launch of their own costs about 5 us, 2% of a V-cycle
// iteration on a 64^3 cell)
// Epilogue at each owned node, with Au the operator result and u_own the
// staged value there:
//   EP_AX       y = Au            (optional FP64 partial of u . Au; with ST_PUPD,
//                                  pout = u_own: the new PCG direction)
//   EP_AXD      y = Au / D        (a power-iteration step: load case 0 of every
//                                  cell, the only one launched)
//   EP_RES      y = b - Au        (optional FP64 partials of r.r, b.u, u.r)
//   EP_PRE      b - Au ; on the fine level restricted to y = P^T (b - Au) on the
//               coarse grid gc, on the coarse levels y = b - Au itself
//   EP_CHEB0    r = b - Au ; dout = r theta_inv / D ; x = u_own
//   EP_CHEB0L   r = b - Au ; x = u_own
//   EP_FIN1     x = u_own + (b - Au) theta_inv / D (a degree-1 smoothing), and
//               with `dot` the FP64 partial of b . x
//   EP_STEP     r = rprev - Au ; dn = c1 u_own + c2 r / D ; dout = dn ;
//               x = xprev + u_own   (xprev = 0 with ST_DSCALE)
//   EP_LAST     the last step: x = xprev + u_own + dn (nothing reads r and d)
//   EP_LASTD    the same with the FP64 partial of b . x (fine level)
// A kernel never writes the vector it stages (neighbours read it), so d/d2 are
// ping-ponged by the caller; x may go over xprev, which only the owner reads.
// Chebyshev coefficients are per sample (each sample's smoother has its own
// spectrum estimate).
#pragma once
#include "kernels.hpp"

namespace femh {

enum Stage : int { ST_PLAIN = 0, ST_DSCALE = 1, ST_PROLONG = 2, ST_PUPD = 3, ST_DPROLONG = 4, ST_PUPDX = 5, ST_RUPD = 6 };
enum Epi : int {
  EP_AX = 0,
  EP_RES = 1,
  EP_CHEB0 = 2,
  EP_STEP = 3,
  EP_PRE = 4,
  EP_FIN1 = 5,
  EP_LAST = 6,
  EP_LASTD = 7,
  EP_AXD = 8,
  EP_CHEB0L = 9
};
constexpr int kMaxCheb = 16;

template <typename T>
struct OpArgs {
  const T *u = nullptr;      // staged vector [R][3][V]
  const T *u2 = nullptr;     // ST_PUPD, ST_PUPDX: previous direction; ST_RUPD: q [R][3][V]
  const double *beta = nullptr;  // ST_PUPD: per-RHS beta [R]
  double *alpha = nullptr;       // per-RHS alpha [R]: read by ST_PUPDX, written by ST_RUPD
  T *pout = nullptr;         // ST_PUPD, ST_PUPDX: staged value written back (new direction); ST_RUPD: r'
  const T *xc = nullptr;     // ST_PROLONG, ST_DPROLONG: coarse vector [R][3][Vc]
  Dims gc{};                 // ST_PROLONG, ST_DPROLONG, fine EP_PRE: coarse dims
  const T *Dinv = nullptr;   // inverse diagonal [B][3][V]
  T *y = nullptr;
  const T *b = nullptr;
  T *r = nullptr;
  const T *rprev = nullptr;
  T *dout = nullptr;
  const T *xprev = nullptr;
  T *x = nullptr;
  const int *act = nullptr;  // [R] activity flags
  Reduce red{};
  int slot = 0;
  int dot = 0;               // EP_RES: r.r -> slot, b.x -> slot2, x.r -> slot3
  int slot2 = 0, slot3 = 0;
  // ST_PUPDX's beta and ST_RUPD's alpha are quotients of two sums of partials,
  // slot2 (np of them) over slot3 (np3); `record` (optional) takes the value at
  // row cnt[r] - ST_PUPDX, cnt the iterations done per RHS
  int np = 0, np3 = 0;
  double *record = nullptr;
  const int *cnt = nullptr;
  // Chebyshev coefficients of this launch, device memory [3][kMaxB]: 1/theta,
  // c1, c2 per sample (null where the variant uses none).  In device memory,
  // not in the arguments, so that a recorded launch sequence stays valid when
  // a new solve brings new spectra.
  const double *cheb = nullptr;
  // outputs stored non-temporally (set by the fine-level launcher for
  // vectors too large to stay in the caches until the next launch reads them)
  int nt = 0;
  // in: the launch is sized for a few remaining right-hand sides; set by the
  // launchers to the workgroup order (work_order in ops.hip)
  int spread = 0;
};

// fine level (tiled cube-mode voxel kernel).  shape: launch shape, bits 0-7
// node planes per workgroup and bits 8-15 the tile variant (TJ x TK owned
// node columns per workgroup: 1 = 16 x 16, 2 = 8 x 32, 3 = 16 x 32); 0 in a
// field is the built-in choice (tiled_default_tile, planes from the grid).
// tiled_parts: partial count of a dot launch with that shape (`fused`: one
// with a fused grid transfer, whose planes come in pairs); tiled_slabs:
// the planes per workgroup actually used (both depend on the element size
// sz, 4 or 8, for a one-cell launch).  ev0/ev1 (optional): events the
// runtime records at the kernel's own start and end (kernel timing).
constexpr int kNumTileShapes = 4;
inline int tiled_shape_code(int tile, int planes) { return (tile << 8) | planes; }
int tiled_default_tile(const Dims &g, int R);  // the tile variant of the built-in shape
template <typename T>
void launch_tiled(int st, int ep, const Dims &g, int R, const T *E, const ModeCoef &mc,
                  const OpArgs<T> &a, hipStream_t s, int shape = 0, hipEvent_t ev0 = nullptr,
                  hipEvent_t ev1 = nullptr);
int tiled_parts(const Dims &g, int R, int shape, int sz, bool fused = false);
int tiled_slabs(const Dims &g, int R, int shape, int sz);
// launch shape for a launch with only Ract of its R right-hand sides active
// (the power iteration: one per cell) and no fused dot: shape's tile, the
// chunk length from the rounds of the active workgroups (shape returned as
// it is when its planes are pinned)
int tiled_sparse_shape(const Dims &g, int R, int Ract, int shape, int sz);

// coarse level (27-point block stencil, one RHS per thread).  cells: the cells
// the launch is sized for (at most R / 6; the others are expected inactive)
template <typename T>
void launch_stencil(int st, int ep, const Dims &g, int R, const T *S, const OpArgs<T> &a,
                    hipStream_t s, int cells);

// x = xn + d
template <typename T>
void launch_add2(int V, int R, const T *xn, const T *d, T *x, const int *act, hipStream_t s);

}  // namespace femh
