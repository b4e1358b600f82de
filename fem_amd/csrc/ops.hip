// ops.hip -- fused operator kernels (see ops.hpp for the staging / epilogue
// contract).  Grids carry the right-hand side q = 6 s + lc; per-sample data
// (moduli, stencils, inverse diagonals, Chebyshev coefficients) is selected
// by s = q / 6.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <atomic>
#include <climits>
#include <cmath>
#include <stdexcept>

#include "device_common.hpp"
#include "ops.hpp"

namespace femh {

// ---------------------------------------------------------------------------
// fine level: tiled cube-mode voxel kernel
//
// K0 = H^T Lambda H per voxel (tables.hpp).  A workgroup owns a TJ x TK tile
// of node columns (j,k) (16 x 16, 8 x 32 or 16 x 32, one thread per column)
// and marches over a chunk of TI planes in i.  Per voxel slab (planes s, s+1):
//   1. node plane s+1 of the tile plus a one-node halo on each j/k side
//      ((TJ+2) x (TK+2) nodes, periodic wrap) is staged into LDS (a
//      two-buffer ring, see below);
//   2. each of the (TJ+1) x (TK+1) voxels touching the tile transforms its
//      top face ((j,k) butterflies; the bottom face is the top face of the
//      slab below, carried in registers), forms the 8 cube modes per
//      component with the i stage, applies the mode coupling scaled by its
//      modulus and splits the result back into bottom- and top-face modes;
//   3. the bottom-face modes plus the top-face modes of the voxel below (the
//      same node plane s) go through one inverse face transform into LDS,
//      and the 4 tile nodes sharing each corner gather them: plane s is
//      complete and passes through the epilogue.
// The j/k halo voxels are recomputed by neighbouring tiles ((TJ+1)(TK+1) /
// (TJ TK) of the voxel work: 1.13 for 16 x 16, 1.10 for 16 x 32) and the i
// halo slab once per chunk ((TI+1)/TI).
constexpr int kTile = 16;
constexpr int kTN = kTile + 2;   // staged nodes per row
constexpr int kTE = kTile + 1;   // voxels per row
constexpr int kEOH = 13;         // LDS stride of one voxel's 12 plane forces (odd: no bank conflicts)

// periodic index for i in [-n, 2n) without a division
__device__ __forceinline__ int wrap1(int i, int n) { return i < 0 ? i + n : (i >= n ? i - n : i); }

// epilogue inputs of one owned node (loaded ahead of the operator work so
// that their latency overlaps it; the set of loads is fixed per variant -- a
// load behind a run-time branch is waited for at the branch's end):
//   EP_RES, EP_PRE: e0 = b ; EP_CHEB0, EP_CHEB0L, EP_FIN1: e0 = b, e1 = 1/D ;
//   EP_STEP, EP_LAST, EP_LASTD: e0 = rprev, e1 = 1/D, e2 = xprev (none from a
//   zero start, ST_DSCALE) ; EP_LASTD: e3 = b (for b . x) ; EP_AXD: e1 = 1/D ;
//   ST_PUPDX: e1 = the old direction, e2 = x
template <typename T>
struct EpiIn {
  T e0[3], e1[3], e2[3], e3[3];
};
__host__ __device__ constexpr bool ep_is_step(int ep) { return ep == EP_STEP || ep == EP_LAST || ep == EP_LASTD; }
__host__ __device__ constexpr bool ep_has_b(int ep) {
  return ep == EP_RES || ep == EP_PRE || ep == EP_CHEB0 || ep == EP_CHEB0L || ep == EP_FIN1;
}

template <typename T, int ST, int EP>
__device__ __forceinline__ void epi_load(const OpArgs<T> &a, const T *__restrict__ Ds, size_t off,
                                         int V, int n, EpiIn<T> &p) {
#pragma unroll
  for (int c = 0; c < 3; c++) {
    const size_t q = off + (size_t)c * V + n;
    if (ep_has_b(EP)) p.e0[c] = a.b[q];
    if (ep_is_step(EP)) p.e0[c] = a.rprev[q];
    if (EP == EP_CHEB0 || EP == EP_FIN1 || ep_is_step(EP) || EP == EP_AXD) p.e1[c] = Ds[(size_t)c * V + n];
    if (ep_is_step(EP)) p.e2[c] = ST == ST_DSCALE ? (T)0 : a.xprev[q];
    if (EP == EP_LASTD) p.e3[c] = a.b[q];
    if (ST == ST_PUPDX) {
      p.e1[c] = a.u2[q];
      p.e2[c] = a.x[q];
    }
  }
}

// FP64 partial sums of the epilogue: EP_AX u.Au ; EP_FIN1, EP_LASTD b.x_new ;
// EP_RES r.r, b.x, x.r (x = the staged vector)
struct DotAcc {
  double a = 0, b = 0, c = 0;
};

// output store of an epilogue; NT: a streaming (non-temporal) store, for
// output vectors far larger than the caches (read back only by a later
// launch, which would find them evicted anyway)
template <bool NT, typename T>
__device__ __forceinline__ void ep_store(T *p, T v) {
  if (NT)
    __builtin_nontemporal_store(v, p);
  else
    *p = v;
}

// epilogue at one owned node (all three components)
template <typename T, int ST, int EP, bool NT = false>
__device__ __forceinline__ void epilogue(const OpArgs<T> &a, const EpiIn<T> &p, T ti, T c1, T c2,
                                         size_t off, int V, int n, const T Au[3], const T uo[3],
                                         DotAcc &dv, T al = 0) {
#pragma unroll
  for (int c = 0; c < 3; c++) {
    const size_t q = off + (size_t)c * V + n;
    if (EP == EP_AX) {
      ep_store<NT>(&a.y[q], Au[c]);
      if (ST == ST_PUPD || ST == ST_PUPDX) ep_store<NT>(&a.pout[q], uo[c]);
      if (ST == ST_PUPDX) ep_store<NT>(&a.x[q], p.e2[c] + al * p.e1[c]);
      if (a.dot) dv.a += (double)uo[c] * (double)Au[c];
    } else if (EP == EP_AXD) {
      ep_store<NT>(&a.y[q], Au[c] * p.e1[c]);
    } else if (EP == EP_RES || EP == EP_PRE) {
      const T rv = p.e0[c] - Au[c];
      ep_store<NT>(&a.y[q], rv);
      if (EP == EP_RES && a.dot) {
        dv.a += (double)rv * (double)rv;
        dv.b += (double)p.e0[c] * (double)uo[c];
        dv.c += (double)uo[c] * (double)rv;
      }
    } else if (EP == EP_FIN1) {
      const T rv = p.e0[c] - Au[c];
      const T xv = uo[c] + rv * ti * p.e1[c];
      ep_store<NT>(&a.x[q], xv);
      if (a.dot) dv.a += (double)p.e0[c] * (double)xv;
    } else if (EP == EP_CHEB0 || EP == EP_CHEB0L) {
      const T rv = p.e0[c] - Au[c];
      ep_store<NT>(&a.r[q], rv);
      if (EP == EP_CHEB0) ep_store<NT>(&a.dout[q], rv * ti * p.e1[c]);
      ep_store<NT>(&a.x[q], uo[c]);
    } else {
      const T rv = p.e0[c] - Au[c];
      const T dn = c1 * uo[c] + c2 * rv * p.e1[c];
      T xv = p.e2[c] + uo[c];
      if (EP != EP_STEP) {
        xv += dn;  // the last step's r and d are not read again
      } else {
        ep_store<NT>(&a.r[q], rv);
        ep_store<NT>(&a.dout[q], dn);
      }
      ep_store<NT>(&a.x[q], xv);
      if (EP == EP_LASTD) dv.a += (double)p.e3[c] * (double)xv;
    }
  }
}

#ifndef FEMH_WAVES64
#define FEMH_WAVES64 1
#endif
constexpr int kWaves64 = FEMH_WAVES64;  // FP64 fine operator: waves per SIMD the registers allow

// Tile shapes (TJ x TK owned node columns per workgroup, TJ*TK threads).
// Launch shape encoding: bits 0-7 node planes per workgroup (0 = built-in),
// bits 8-15 tile variant (0 = built-in, tiled_default_tile).
struct TileShape {
  int tj, tk;
};
constexpr TileShape kTileShapes[kNumTileShapes] = {{16, 16}, {16, 16}, {8, 32}, {16, 32}};

// The built-in tile on grids whose z extent is a multiple of 32 (and y of
// 16) and at least 64:
//  * batched launches (24 or more right-hand sides): 16 x 32 -- a tile row is
//    a whole 128-byte line in FP32 and the j/k halo recompute drops from 1.13
//    to 1.10 (64^3, 16 cells: 15% less time than 16 x 16 over the four
//    variants of a PCG iteration);
//  * one cell (6 right-hand sides, too few workgroups for the larger tile):
//    8 x 32 -- as many tiles as 16 x 16, so as many workgroups, with
//    whole-line rows (64^3: 53.3 -> 50.8 us per FP64 launch, 31.2 -> 28.8 us
//    per FP32 launch).
// Smaller or odd grids (the 24^3 and 48^3 cells of an uneven batch, which
// waste less on partial tiles) keep 16 x 16.
int tiled_default_tile(const Dims &g, int R) {
  if (g.nz >= 64 && g.nz % 32 == 0 && g.ny % 16 == 0) return R >= 24 ? 3 : (R <= kRHS ? 2 : 1);
  return 1;
}

static inline TileShape tile_of(const Dims &g, int R, int shape) {
  int v = (shape >> 8) & 0xff;
  if (v <= 0 || v >= kNumTileShapes) v = tiled_default_tile(g, R);
  return kTileShapes[v];
}

static inline int tiled_tiles(const Dims &g, const TileShape &ts) {
  return ((g.ny + ts.tj - 1) / ts.tj) * ((g.nz + ts.tk - 1) / ts.tk);
}

static int tiled_resident(int sz, const TileShape &ts);

// Launches with a fused grid transfer (`fused`) have chunks of an even length,
// so that a chunk holds whole coarse planes; the others may take odd ones (a
// 16^3 cell: one plane per workgroup).
static inline int even_chunk(int ti, bool fused) { return fused ? ti + (ti & 1) : ti; }

// Chunk length for a launch whose active workgroups (Ract active right-hand
// sides) fill the device about once or less: the rounds of resident
// workgroups set the time, so take the length that minimises rounds x slabs
// per workgroup (at most 255 planes, the width of the launch-shape field).
static int round_chunk(const Dims &g, const TileShape &ts, int tiles, int Ract, int sz, bool fused = false) {
  const long res = tiled_resident(sz, ts);
  long best = LONG_MAX;
  int TI = g.nx;
  for (int c = (g.nx + 253) / 254; c <= g.nx; c++) {
    const int ti = even_chunk((g.nx + c - 1) / c, fused), ch = (g.nx + ti - 1) / ti;
    if ((long)tiles * ch > kMaxPartials) continue;
    const long rounds = ((long)tiles * ch * Ract + res - 1) / res, cost = rounds * (ti + 1);
    if (cost < best) {
      best = cost;
      TI = ti;
    }
  }
  return TI;
}

static inline int tiled_chunk(const Dims &g, int R, int shape, int sz, bool fused = false) {
  const TileShape ts = tile_of(g, R, shape);
  const int tiles = tiled_tiles(g, ts);
  const int want = shape & 0xff;
  // planes per chunk: `want` when given (an autotuned shape).  One cell (six
  // right-hand sides) gives too few workgroups to fill the device more than
  // about once, so the rounds of resident workgroups set the time: take the
  // chunk length that minimises rounds x slabs per workgroup (64^3 in FP64:
  // 13 planes, 480 workgroups in one round, against 8 planes and 768
  // workgroups in two).  Batches: about 32 planes (halo slab overhead 1/32)
  // but enough chunks to put ~2 workgroups of 256 threads per CU across the
  // right-hand sides.  At most kMaxPartials workgroups per right-hand side
  // either way.
  int TI = 32;
  if (want > 0) {
    TI = want;
  } else if (R <= kRHS) {
    TI = round_chunk(g, ts, tiles, R, sz, fused);
  } else {
    while (TI > 2 && (long)tiles * ((g.nx + TI - 1) / TI) * R * ts.tj * ts.tk < 512L * 256) TI /= 2;
  }
  if (TI > g.nx) TI = g.nx;
  TI = even_chunk(TI, fused);
  while ((long)tiles * ((g.nx + TI - 1) / TI) > kMaxPartials) TI = even_chunk(TI + 1, fused);
  return TI;
}

int tiled_slabs(const Dims &g, int R, int shape, int sz) { return tiled_chunk(g, R, shape, sz); }

int tiled_sparse_shape(const Dims &g, int R, int Ract, int shape, int sz) {
  if (shape & 0xff) return shape;  // planes pinned (autotuned or set)
  int v = (shape >> 8) & 0xff;
  if (v <= 0 || v >= kNumTileShapes) v = tiled_default_tile(g, R);
  const TileShape ts = kTileShapes[v];
  return tiled_shape_code(v, round_chunk(g, ts, tiled_tiles(g, ts), Ract, sz));
}

int tiled_parts(const Dims &g, int R, int shape, int sz, bool fused) {
  const int TI = tiled_chunk(g, R, shape, sz, fused);
  return tiled_tiles(g, tile_of(g, R, shape)) * ((g.nx + TI - 1) / TI);
}

// Workgroups are dispatched round-robin over the 8 XCDs (workgroup b to XCD
// b mod 8), each with its own L2.  xcd_order maps the dispatch index to a
// logical index so that every XCD runs one contiguous range of logical
// workgroups: consecutive logical workgroups -- which share halo rows and
// per-cell data -- then meet in the same L2.
__device__ __forceinline__ int xcd_order(int b, int n) {
  const int x = b & 7, slot = b >> 3, per = n >> 3, rem = n & 7;
  return x * per + (x < rem ? x : rem) + slot;
}

// Work of a launch as (cell, unit, inner): `inner` workgroups share a unit's data
// (load cases or their groups) and neighbouring units (tiles and planes of a
// cell) share halos.  Two logical orders:
//  * cell, unit, inner: neighbouring units follow each other on one XCD, but a
//    cell lies on one or two XCDs, so the launches of a batch's last cells run
//    there alone (48^3, one of 12 cells left: 65 us a fine launch of 324 active
//    workgroups);
//  * spread: eighth of the units, cell, unit within the eighth, inner: every
//    XCD gets an eighth of every cell (that launch: 24 us).
// Spread is taken for launches sized for a few remaining right-hand sides
// (live_rhs), and where every eighth is the same number of equal units and
// large enough for neighbours to share their halos:
//  * the units divide by eight; otherwise an XCD has up to twice another's work
//    (40^3 in FP64, 18 units: 33.2 -> 39.3 ms);
//  * fine launches: chunks of one length.  A shorter last chunk lies on the
//    same XCDs for every cell (chunks of 32 and 8 planes, 16 cells of 40 x 64 x
//    96 in mixed precision: 1.19 times the time; 24^3, 16 + 8: 1.13 in FP64;
//    48 x 64 x 64, 32 + 16: 1.09; 56^3, 32 + 24: 1.05);
//  * at least two fine units per eighth (one: 32^3, 16 cells: 1.06) and eight
//    stencil units (two, the level of 32^3: 1.02; ten or twelve, the levels of
//    40^3 and 48^3: 1.00-1.01 where all cells take as long, but 0.98 in an uneven
//    batch of 64 binary cells, whose cells converge one after the other).
// Within these it cost no more than the 1% to which runs agree, but for 1.6%
// on 4 cells of 32 x 64 x 128 in mixed precision; 64^3 0.97-0.99, 80^3 and 96^3
// 0.99, 64 x 96 x 64 0.94, 128 x 64 x 64 0.95-0.98, 32 x 64 x 128 in FP64 0.95 of
// the time.
constexpr int kSpreadFine = 16, kSpreadStencil = 64;  // least units
static inline int spread_rule(int sparse, int units, int least, bool equal) {
  return sparse || (units % 8 == 0 && units >= least && equal);
}
struct WorkId {
  int cell, unit, inner;
};
__device__ __forceinline__ WorkId work_order(int b, int n, int cells, int units, int inner, int spread) {
  const int L = xcd_order(b, n);
  if (!spread) return {L / (inner * units), L / inner % units, L % inner};
  const int q = L / (inner * cells);  // units before this workgroup's, all cells alike
  int p = q * 8 / units;              // its eighth: units [p U / 8, (p + 1) U / 8)
  while ((p + 1) * units / 8 <= q) p++;
  const int u0 = p * units / 8, su = (p + 1) * units / 8 - u0;
  const int rem = L - u0 * inner * cells, t = rem / inner;
  return {t / su, u0 + t % su, rem - t * inner};
}

// raw buffer access: base pointer and byte range in a resource, one 32-bit
// lane offset plus a scalar offset per access (no 64-bit address arithmetic)
__device__ __forceinline__ __amdgpu_buffer_rsrc_t brsrc(const void *p, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void *)p, (short)0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ float bload(__amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff, float *) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
}
__device__ __forceinline__ double bload(__amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff, double *) {
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0));
}

// grid: one dimension of tiles * chunks * R workgroups, units of (chunk, tile)
// with the six load cases of a tile (same moduli and diagonal) next to each
// other on one XCD (work_order).
//
// LDS: staged node planes in a two-buffer ring, node-interleaved
// (up[buf][3 * slot + c]), so that the 12 values of a voxel face and the
// owned node's value are immediate offsets from one address; eo holds each
// voxel's 12 bottom-face forces (odd stride: no bank conflicts).  A buffer is
// overwritten two slabs after it was filled, behind the barrier that closes
// the slab in between (every read of it -- the FP64 bottom face, the owned
// node's staged value -- happens before that barrier).
//
// Grid transfers inside the kernel: as passes of their own they moved three more
// vectors, and the launches around them one more each, at 4.2-4.6 of the 4.85
// TB/s that a large copy reaches.  64^3, 16 cells in FP32: pre-smoothing 297 us
// and restriction 92 us became one launch of 282 us, prolongation 106 us and
// post-smoothing 227 us one of 285 us; these launches keep the VALU 62-63% busy,
// and that, not the vectors, is what bounds them.
//  * RS (EP_PRE): the residual goes to the coarse right-hand side and never to
//    memory.  The tile computes one more node row and column at its low j and
//    k sides (and its chunk one more plane), so that every coarse node above
//    its owned nodes has the 27 residuals of its full weighting in the
//    workgroup; they pass through rb in LDS, plane by plane, and each coarse
//    node's sum is carried in FP64 by one thread.
//  * ST_PROLONG / ST_DPROLONG: the staged value is x + P xc, x read (PROLONG)
//    or formed as b / (theta D) (DPROLONG: the degree-1 pre-smoothing, whose x
//    is then never stored).  The coarse nodes around the tile are staged into
//    cl one coarse plane at a time, two slabs ahead; each staging slot keeps
//    its interpolated value of the lower coarse plane.
//  * Residual update (RUPD): r' = r - alpha q is formed where it is staged,
//    (theta D)^-1 r' goes to the staged plane and r' itself to rb, whose three
//    planes rotate: one being staged, one turned into the residual in place, one
//    being restricted.
// Waves per SIMD the FP32 variants are compiled for: 4 (at most 128 VGPRs);
// three where the 256-thread tiles' LDS lets no fourth workgroup in (RUPD).
template <typename T, int ST, int NT>
constexpr int tiled_waves() {
  return sizeof(T) != 4 ? kWaves64 : ST == ST_RUPD && NT < 512 ? 3 : 4;
}

template <typename T, int ST, int EP, int TJ, int TK, bool RS>
__global__ __launch_bounds__(TJ * TK, (tiled_waves<T, ST, TJ * TK>())) void k_tiled(Dims g, const T *__restrict__ E,
                                                                           ModeC<T> mc, OpArgs<T> a, int TI,
                                                                           int tiles_k, int tiles, int chunks) {
  constexpr int NT = TJ * TK;                           // threads = owned nodes per plane
  constexpr int H = RS ? 1 : 0;                         // extra node row / column / plane at the low sides
  constexpr int NJ = TJ + 2 + H, NK = TK + 2 + H, NS = NJ * NK;  // staged nodes (one-node halo)
  constexpr int EJ = TJ + 1 + H, EK = TK + 1 + H, NE = EJ * EK;  // voxels touching the tile
  constexpr int QS = (NS + NT - 1) / NT, QE = (NE + NT - 1) / NT;
  static_assert(NT % 64 == 0 && QS <= 2 && QE <= 2, "tile shape");
  constexpr bool kProl = ST == ST_PROLONG || ST == ST_DPROLONG;
  constexpr bool kStD = ST == ST_DSCALE || ST == ST_DPROLONG || ST == ST_RUPD;  // stages b / (theta D)
  constexpr bool kPupd = ST == ST_PUPD || ST == ST_PUPDX, kRupd = ST == ST_RUPD;
  static_assert(!kRupd || RS, "the residual update stages for the restricted residual");
  constexpr int CJ = TJ / 2 + 2, CK = TK / 2 + 2;              // coarse nodes around the tile (kProl)
  constexpr unsigned SZ = sizeof(T);
  const int inner = EP == EP_AXD ? 1 : kRHS;  // (the power iteration runs load case 0 only)
  const WorkId id = work_order(blockIdx.x, gridDim.x, gridDim.x / (inner * tiles * chunks), tiles * chunks, inner, a.spread);
  const int smp = id.cell, tile = id.unit % tiles, chunk = id.unit / tiles;
  const int r = smp * kRHS + id.inner;
  if (!a.act[r]) return;
  const int V = g.V;
  const unsigned VB = (unsigned)V * SZ;  // bytes per component plane
  const __amdgpu_buffer_rsrc_t rE = brsrc(E + (size_t)smp * V, VB);
  const T *__restrict__ Ds = a.Dinv ? a.Dinv + (size_t)smp * 3 * V : nullptr;
  const size_t off = (size_t)r * 3 * V;
  const __amdgpu_buffer_rsrc_t rU = brsrc(a.u + off, 3 * VB);
  const __amdgpu_buffer_rsrc_t rU2 = brsrc(kPupd || kRupd ? a.u2 + off : a.u + off, 3 * VB);
  const __amdgpu_buffer_rsrc_t rD = brsrc(Ds ? Ds : a.u + off, 3 * VB);
  const T ti = a.cheb ? (T)a.cheb[smp] : (T)0, c1 = a.cheb ? (T)a.cheb[kMaxB + smp] : (T)0,
          c2 = a.cheb ? (T)a.cheb[2 * kMaxB + smp] : (T)0;
  T bt = ST == ST_PUPD ? (T)a.beta[r] : (T)0, al = ST == ST_PUPDX ? (T)a.alpha[r] : (T)0;
  if constexpr (ST == ST_PUPDX || kRupd) {
    const double num = sum_parts_wave(a.red, a.slot2, r, a.np), den = sum_parts_wave(a.red, a.slot3, r, a.np3);
    const double v = den != 0.0 ? num / den : 0.0;
    (kRupd ? al : bt) = (T)v;
    if (id.unit == 0 && threadIdx.x == 0) {
      if (kRupd) a.alpha[r] = v;
      if (a.record) a.record[(size_t)(a.cnt[r] - (kRupd ? 0 : 1)) * kMaxR + r] = v;
    }
  }
  __shared__ T up[2][3 * NS];
  __shared__ T eo[NE * kEOH];
  __shared__ T cl[kProl ? 3 * CJ * CK : 1];
  // (kRupd: plane ip's r' waits in part (ip - i0) mod 3 from its staging until the
  // gather turns it into the residual in place, and that until its restriction)
  constexpr int RP = 3 * (TJ + 1) * (TK + 1);
  __shared__ T rb[RS ? (kRupd ? 3 : 1) * RP : 1];
  const int tid = threadIdx.x;
  // staging slots and voxels go to threads in an order rotated by a wave per
  // workgroup, so that the second round of the extra ones does not fall on
  // the same wave -- hence the same SIMD -- in every workgroup; owned nodes
  // (the epilogue) keep the plain thread order
  const int vt = (tid + 64 * ((int)(blockIdx.x >> 3) & (NT / 64 - 1))) & (NT - 1);
  const int j0 = (tile / tiles_k) * TJ, k0 = (tile % tiles_k) * TK;
  const int i0 = chunk * TI;
  const int iend = min(i0 + TI, g.nx);
  const int plane = g.ny * g.nz;

  // per-thread staging slots (fixed across planes): node offsets in a plane
  int soff[QS];
#pragma unroll
  for (int q = 0; q < QS; q++) {
    const int t = vt + q * NT;
    soff[q] = -1;
    if (t < NS) {
      const int nj = t / NK, nk = t - nj * NK;
      // slots of a tile wider than the grid wrap more than once
      const int jj = ((j0 - 1 - H + nj) % g.ny + g.ny) % g.ny, kk = ((k0 - 1 - H + nk) % g.nz + g.nz) % g.nz;
      soff[q] = jj * g.nz + kk;
    }
  }
  // per-thread voxels (fixed across slabs): modulus offsets in a plane
  int eoff[QE];
#pragma unroll
  for (int q = 0; q < QE; q++) {
    const int e = vt + q * NT;
    eoff[q] = -1;
    if (e < NE) {
      const int ej = e / EK, ek = e - ej * EK;
      const int jj = ((j0 - 1 - H + ej) % g.ny + g.ny) % g.ny, kk = ((k0 - 1 - H + ek) % g.nz + g.nz) % g.nz;
      eoff[q] = jj * g.nz + kk;
    }
  }

  // Coarse nodes of the fused prolongation: thread t < CJ CK brings node
  // (j0/2 - 1 + t / CK, k0/2 - 1 + t % CK) of a coarse plane from memory (cfetch,
  // two slabs ahead) to cl (cput).  A slot's 2D value (interp) adds two rows of
  // two columns with weights (1, 0) at even and (1/2, 1/2) at odd fine nodes.
  // (the interpolated value of the lower coarse plane: a thread's first slot
  // keeps it in registers, the second slots in LDS, as with the voxels below)
  constexpr int NSX = NS > NT ? NS - NT : 1;
  __shared__ T ic[kProl ? 3 * NSX : 1];
  T cr[3], ia[3];
  unsigned coff = 0;
  __amdgpu_buffer_rsrc_t rC = rU;
  unsigned CB = 0;
  if constexpr (kProl) {
    CB = (unsigned)a.gc.V * SZ;
    rC = brsrc(a.xc + (size_t)r * 3 * a.gc.V, 3 * CB);
    const int cj = ((j0 / 2 - 1 + tid / CK) % a.gc.ny + a.gc.ny) % a.gc.ny,
              ck = ((k0 / 2 - 1 + tid % CK) % a.gc.nz + a.gc.nz) % a.gc.nz;
    coff = (unsigned)(cj * a.gc.nz + ck);
  }
  auto cfetch = [&](int I) {
    if (tid < CJ * CK) {
      const unsigned vo = ((unsigned)(wrap1(I, a.gc.nx) * a.gc.ny * a.gc.nz) + coff) * SZ;
#pragma unroll
      for (int c = 0; c < 3; c++) cr[c] = bload(rC, vo, c * CB, (T *)nullptr);
    }
  };
  auto cput = [&]() {
    if (tid < CJ * CK) {
#pragma unroll
      for (int c = 0; c < 3; c++) cl[3 * tid + c] = cr[c];
    }
  };
  // slot (nj, nk) is fine node (j0 - 1 + nj, k0 - 1 + nk): odd where nj is even.
  // Its place in cl and its parities are packed in one register, which passes
  // through an empty asm so that what derives from it is formed where it is
  // used instead of being kept in seven registers over the loop.
  int cpk[QS];
#pragma unroll
  for (int q = 0; q < QS; q++) {
    const int t = vt + q * NT, nj = t / NK, nk = t - nj * NK;
    cpk[q] = (3 * (((nj + 1) >> 1) * CK + ((nk + 1) >> 1))) << 2 | (nj & 1) << 1 | (nk & 1);
  }
  auto interp = [&](int q, T (&v)[3]) {
    int pk = cpk[q];
    asm volatile("" : "+v"(pk));
    const T *row0 = cl + (pk >> 2);
    const int dj = (pk & 2) ? 0 : 3 * CK, dk = (pk & 1) ? 0 : 3;
    const T wj0 = (pk & 2) ? (T)1 : (T)0.5, wj1 = (pk & 2) ? (T)0 : (T)0.5;
    const T wk0 = (pk & 1) ? (T)1 : (T)0.5, wk1 = (pk & 1) ? (T)0 : (T)0.5;
#pragma unroll
    for (int c = 0; c < 3; c++) {
      const T s0 = wk0 * row0[c] + wk1 * row0[dk + c], s1 = wk0 * row0[dj + c] + wk1 * row0[dj + dk + c];
      v[c] = wj0 * s0 + wj1 * s1;
    }
  };

  // staging of node plane ip into LDS buffer buf, software-pipelined: fetch()
  // issues the loads of a plane into registers one slab ahead, put() scales
  // and stores them.
  T pf[QS][3], pd[QS][3], pq[kRupd ? QS : 1][3];
  auto fetch = [&](int ip) {
    const int iw = wrap1(ip, g.nx);
#pragma unroll
    for (int q = 0; q < QS; q++) {
      if (soff[q] < 0) continue;
      const unsigned vo = (unsigned)(iw * plane + soff[q]) * SZ;
#pragma unroll
      for (int c = 0; c < 3; c++) {
        pf[q][c] = bload(rU, vo, c * VB, (T *)nullptr);
        if (kStD) pd[q][c] = bload(rD, vo, c * VB, (T *)nullptr);
        if (kPupd) pd[q][c] = bload(rU2, vo, c * VB, (T *)nullptr);
        if constexpr (kRupd) pq[q][c] = bload(rU2, vo, c * VB, (T *)nullptr);
      }
    }
  };
  int part = 0;  // kRupd: offset in rb of the plane the slab completes
  auto put = [&](int buf, int ip) {
#pragma unroll
    for (int q = 0; q < QS; q++) {
      if (soff[q] < 0) continue;
      T *dst = &up[buf][3 * (vt + q * NT)];
      T v[3];
      if constexpr (kRupd) {
#pragma unroll
        for (int c = 0; c < 3; c++) pf[q][c] = pf[q][c] - al * pq[q][c];
        // place of the staged node among the owned and extra ones, derived anew
        // (not kept over the loop; see cpk)
        int t = vt + q * NT;
        asm volatile("" : "+v"(t));
        const int sj = t / NK - 1, sk = t - (sj + 1) * NK - 1;
        if (sj >= 0 && sj <= TJ && sk >= 0 && sk <= TK) {
          T *up1 = rb + (part == 2 * RP ? 0 : part + RP);
#pragma unroll
          for (int c = 0; c < 3; c++) up1[(c * (TJ + 1) + sj) * (TK + 1) + sk] = pf[q][c];
        }
      }
#pragma unroll
      for (int c = 0; c < 3; c++)
        v[c] = kStD ? pf[q][c] * (ti * pd[q][c]) : kPupd ? pf[q][c] + bt * pd[q][c] : pf[q][c];
      if constexpr (kProl) {
        // (x is rounded before the correction is added, as when it is stored)
#pragma clang fp contract(off)
        T *ix = ic + (vt + q * NT - NT);  // (second slots only)
        if (ip & 1) {
          T ib[3];
          interp(q, ib);
#pragma unroll
          for (int c = 0; c < 3; c++) {
            v[c] = v[c] + (T)0.5 * ((q == 0 ? ia[c] : ix[c * NSX]) + ib[c]);
            if (q == 0)
              ia[c] = ib[c];
            else
              ix[c * NSX] = ib[c];
          }
        } else {
#pragma unroll
          for (int c = 0; c < 3; c++) v[c] = v[c] + (q == 0 ? ia[c] : ix[c * NSX]);
        }
      }
#pragma unroll
      for (int c = 0; c < 3; c++) dst[c] = v[c];
    }
  };

  const int nj = tid / TK, nk = tid % TK;  // owned node, output tile coords
  const int gj = j0 + nj, gk = k0 + nk;
  const bool owns = (gj < g.ny) && (gk < g.nz);
  const int ot = 3 * ((nj + 1 + H) * NK + nk + 1 + H);  // owned node in the staged plane
  // RS: the extra nodes, row j0 - 1 (k0 - 1 ..) and column k0 - 1 (j0 ..)
  const int xa = tid <= TK ? 0 : tid - TK, xb = tid <= TK ? tid : 0;
  const bool extra = RS && tid < TJ + TK + 1;
  unsigned xoff = 0;
  if constexpr (RS) {
    const int jj = ((j0 - 1 + xa) % g.ny + g.ny) % g.ny, kk = ((k0 - 1 + xb) % g.nz + g.nz) % g.nz;
    xoff = (unsigned)(jj * g.nz + kk);
  }
  const __amdgpu_buffer_rsrc_t rB = brsrc(RS ? a.b + off : a.u + off, 3 * VB);
  double racc = 0;  // RS: this thread's coarse node sum
  // RS: restriction of residual plane ip in rb: rows and columns with weights
  // 1/2, 1, 1/2, planes 2I - 1, 2I, 2I + 1 into coarse plane I
  auto restrict_plane = [&](int ip, int at) {
    constexpr int CN = (TJ / 2) * (TK / 2);
    if (tid >= 3 * CN) return;
    const int c = tid / CN, q = tid - c * CN, J = q / (TK / 2), K = q - J * (TK / 2);
    const T *p = rb + at + c * (TJ + 1) * (TK + 1) + 2 * J * (TK + 1) + 2 * K;
    double s = 0;
#pragma unroll
    for (int oj = 0; oj < 3; oj++) {
      const T *row = p + oj * (TK + 1);
      const double rs = 0.5 * (double)row[0] + (double)row[1] + 0.5 * (double)row[2];
      s += (oj == 1 ? 1.0 : 0.5) * rs;
    }
    if (ip & 1) {
      const int I = (ip - 1) >> 1, gJ = j0 / 2 + J, gK = k0 / 2 + K;
      if (ip > i0 && gJ < a.gc.ny && gK < a.gc.nz)
        a.y[((size_t)r * 3 + c) * a.gc.V + ((size_t)I * a.gc.ny + gJ) * a.gc.nz + gK] = (T)(racc + 0.5 * s);
      racc = 0.5 * s;
    } else {
      racc = racc + s;
    }
  };
  DotAcc dv;

  // Per voxel (three components, corners v = 4 bi + 2 bj + bk) the cube-mode
  // transform is separable: the (j,k) transform of each face, then the i
  // stage.  A voxel's top face is the bottom face of the voxel above, so
  // its transformed values are carried to the next slab (FP32; FP64 would
  // spend too many registers and transforms the bottom face again).  On the
  // way back, the i stage splits the modal forces into a bottom and a top
  // face; the top face of slab s-1 and the bottom face of slab s lie on the
  // same node plane s, so they are summed before one inverse face transform
  // -- plane s is then complete after a single LDS exchange.
  // A thread's first voxel keeps these values in registers; the few second
  // ones (NE - NT of the tile) keep theirs in LDS, where only their own thread
  // touches them: in registers they would cost every thread 24.
  constexpr bool kReuse = sizeof(T) == 4;
  constexpr int NX = NE > NT ? NE - NT : 1;
  __shared__ T carry[(kReuse ? 24 : 12) * NX];
  T ftop[3][4], tmod[3][4];
  auto face_load = [&](int buf, int ej, int ek, T (&f)[3][4]) {
    const T *src = &up[buf][3 * (ej * NK + ek)];
#pragma unroll
    for (int v = 0; v < 4; v++)
#pragma unroll
      for (int c = 0; c < 3; c++) f[c][v] = src[3 * ((v >> 1) * NK + (v & 1)) + c];
  };
  // forward (j,k) transform per axis: (a, b) -> (a + b, b - a)
  auto face_fwd = [](T (&f)[3][4]) {
#pragma unroll
    for (int c = 0; c < 3; c++)
#pragma unroll
      for (int mb = 2; mb >= 1; mb >>= 1)
#pragma unroll
        for (int v = 0; v < 4; v++)
          if (!(v & mb)) {
            const T a0 = f[c][v], b0 = f[c][v | mb];
            f[c][v] = a0 + b0;
            f[c][v | mb] = b0 - a0;
          }
  };
  // inverse (j,k) transform per axis: (a, b) -> (a - b, a + b)
  auto face_inv = [](T (&f)[3][4]) {
#pragma unroll
    for (int c = 0; c < 3; c++)
#pragma unroll
      for (int mb = 2; mb >= 1; mb >>= 1)
#pragma unroll
        for (int v = 0; v < 4; v++)
          if (!(v & mb)) {
            const T a0 = f[c][v], b0 = f[c][v | mb];
            f[c][v] = a0 - b0;
            f[c][v | mb] = a0 + b0;
          }
  };

  if constexpr (kProl) {
    // (i0 is even: the first staged plane, i0 - 1, lies between coarse planes
    // i0/2 - 1 and i0/2)
    cfetch(i0 / 2 - 1);
    cput();
    __syncthreads();
#pragma unroll
    for (int q = 0; q < QS; q++) {
      if (soff[q] < 0) continue;
      T v[3];
      interp(q, v);
#pragma unroll
      for (int c = 0; c < 3; c++) {
        if (q == 0)
          ia[c] = v[c];
        else
          ic[c * NSX + vt + q * NT - NT] = v[c];
      }
    }
    cfetch(i0 / 2);
    __syncthreads();
    cput();
    cfetch(i0 / 2 + 1);
    __syncthreads();
  }
  fetch(i0 - 1 - H);
  put(0, i0 - 1 - H);
  fetch(i0 - H);
  for (int sl = i0 - 1 - H, p = 0; sl < iend; sl++, p++, part = !kRupd ? 0 : part == 2 * RP ? 0 : part + RP) {
    const int cur = p & 1, nxt = cur ^ 1;
    const int sw = wrap1(sl, g.nx);
    // loads in the order they are consumed: moduli of this slab, epilogue
    // inputs of plane sl, then plane sl + 2 for the next slab
    T Ev[QE];
#pragma unroll
    for (int q = 0; q < QE; q++)
      Ev[q] = eoff[q] >= 0 ? bload(rE, (unsigned)(sw * plane + eoff[q]) * SZ, 0u, (T *)nullptr) : (T)0;
    const size_t nown = (size_t)sw * plane + gj * g.nz + gk;
    EpiIn<T> pin;
    if ((EP != EP_AX || ST == ST_PUPDX) && !kRupd && p > 0 && owns)
      epi_load<T, ST, EP>(a, Ds, off, V, (int)nown, pin);
    T xin[3];
    if constexpr (RS && !kRupd) {
      if (p > 0 && extra) {
#pragma unroll
        for (int c = 0; c < 3; c++)
          xin[c] = bload(rB, ((unsigned)(sw * plane) + xoff) * SZ, c * VB, (T *)nullptr);
      }
    }
    put(nxt, sl + 1);
    if (sl + 2 <= iend) fetch(sl + 2);
    // (this buffer was last read before the barrier that closed the previous
    // slab; the previous slab's gather of eo is behind that barrier too)
    __syncthreads();
    if constexpr (RS) {
      if (p > 1) restrict_plane(sl - 1, !kRupd ? 0 : part == 0 ? 2 * RP : part - RP);
    }
    if constexpr (kProl) {
      // (the odd plane that reads cl is put in the next slab)
      if (!(p & 1)) {
        cput();
        cfetch((sl + 1) / 2 + 2);
      }
    }
    if constexpr (kRupd) {
      if (p > 0 && sl >= i0 && owns) {
#pragma unroll
        for (int c = 0; c < 3; c++) {
          const T v = rb[part + (c * (TJ + 1) + nj + 1) * (TK + 1) + nk + 1];
          if (a.nt)
            ep_store<true>(&a.pout[off + (size_t)c * V + nown], v);
          else
            ep_store<false>(&a.pout[off + (size_t)c * V + nown], v);
          dv.a += (double)v * (double)v;
        }
      }
    }
    T uo[3];
    if (EP != EP_PRE && p > 0 && owns) {
#pragma unroll
      for (int c = 0; c < 3; c++) uo[c] = up[cur][ot + c];
    }
#pragma unroll
    for (int q = 0; q < QE; q++) {
      if (eoff[q] < 0) continue;
      int e = vt + q * NT;
      if (kRupd && q > 0) asm volatile("" : "+v"(e));  // (second voxels: addresses not kept over the loop)
      const int ej = e / EK, ek = e - ej * EK;
      T fb[3][4], ft[3][4];
      face_load(nxt, ej, ek, ft);
      face_fwd(ft);
      T *cy = carry + (e - NT);  // (second voxels only)
      if (kReuse && p > 0) {
#pragma unroll
        for (int c = 0; c < 3; c++)
#pragma unroll
          for (int v = 0; v < 4; v++) fb[c][v] = q == 0 ? ftop[c][v] : cy[(12 + 4 * c + v) * NX];
      } else {
        face_load(cur, ej, ek, fb);
        face_fwd(fb);
      }
      if (kReuse) {
#pragma unroll
        for (int c = 0; c < 3; c++)
#pragma unroll
          for (int v = 0; v < 4; v++) {
            if (q == 0)
              ftop[c][v] = ft[c][v];
            else
              cy[(12 + 4 * c + v) * NX] = ft[c][v];
          }
      }
      // i stage: modes sm = 4 si + s_jk
      T w[3][8];
#pragma unroll
      for (int c = 0; c < 3; c++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
          w[c][v] = fb[c][v] + ft[c][v];
          w[c][4 + v] = ft[c][v] - fb[c][v];
        }
      // coupling and inverse i stage: bottom-face (plane sl) and top-face
      // (plane sl+1) modal forces.  FP64 folds the two per component (fewer
      // live registers); FP32 keeps them apart, which schedules without
      // spills at 4 waves per SIMD
      T bm[3][4], tm[3][4];
#pragma unroll
      for (int c = 0; c < 3; c++)
#pragma unroll
        for (int v = 0; v < 4; v++) tm[c][v] = q == 0 ? tmod[c][v] : cy[(4 * c + v) * NX];
      if constexpr (sizeof(T) == 8) {
        couple_split<T>(w, Ev[q], mc, bm, tm, p > 0);
      } else {
        T z[3][8];
        mode_couple<T>(w, Ev[q], mc, z);
#pragma unroll
        for (int c = 0; c < 3; c++)
#pragma unroll
          for (int v = 0; v < 4; v++) {
            bm[c][v] = z[c][v] - z[c][4 + v];
            if (p > 0) bm[c][v] += tm[c][v];
            tm[c][v] = z[c][v] + z[c][4 + v];
          }
      }
#pragma unroll
      for (int c = 0; c < 3; c++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
          if (q == 0)
            tmod[c][v] = tm[c][v];
          else
            cy[(4 * c + v) * NX] = tm[c][v];
        }
      if (p > 0) {
        face_inv(bm);
        T *dst = eo + e * kEOH;
#pragma unroll
        for (int v = 0; v < 4; v++)
#pragma unroll
          for (int c = 0; c < 3; c++) dst[3 * v + c] = bm[c][v];
      }
    }
    // the first slab completes no plane (uniform branch); its buffer is read above
    // and refilled by the next slab's put, so the slab still closes with a
    // barrier
    __syncthreads();
    if (p == 0) continue;
    // plane sl: voxel columns (a+dj, b+dk) hold this node as face corner
    // (1-dj, 1-dk)
    auto gather = [&](int na, int nb, T (&Au)[3]) {
#pragma unroll
      for (int c = 0; c < 3; c++) Au[c] = 0;
#pragma unroll
      for (int dj = 0; dj < 2; dj++)
#pragma unroll
        for (int dk = 0; dk < 2; dk++) {
          const T *src = eo + ((na + dj) * EK + nb + dk) * kEOH + 3 * (2 * (1 - dj) + (1 - dk));
#pragma unroll
          for (int c = 0; c < 3; c++) Au[c] += src[c];
        }
    };
    if constexpr (RS) {
      T Au[3];
      if (owns) {
        gather(nj + 1, nk + 1, Au);
#pragma unroll
        for (int c = 0; c < 3; c++) {
          T *at = rb + part + (c * (TJ + 1) + nj + 1) * (TK + 1) + nk + 1;
          *at = (kRupd ? *at : pin.e0[c]) - Au[c];
        }
      }
      if (extra) {
        int x = tid;
        if (kRupd) asm volatile("" : "+v"(x));  // (addresses not kept over the loop)
        const int ya = x <= TK ? 0 : x - TK, yb = x <= TK ? x : 0;
        gather(ya, yb, Au);
#pragma unroll
        for (int c = 0; c < 3; c++) {
          T *at = rb + part + (c * (TJ + 1) + ya) * (TK + 1) + yb;
          *at = (kRupd ? *at : xin[c]) - Au[c];
        }
      }
    } else if (owns) {
      T Au[3];
      gather(nj, nk, Au);
      if (a.nt)  // (one uniform branch per node, not per store)
        epilogue<T, ST, EP, true>(a, pin, ti, c1, c2, off, V, (int)nown, Au, uo, dv, al);
      else
        epilogue<T, ST, EP, false>(a, pin, ti, c1, c2, off, V, (int)nown, Au, uo, dv, al);
    }
  }
  if constexpr (RS) {
    __syncthreads();
    restrict_plane(iend - 1, !kRupd ? 0 : part == 0 ? 2 * RP : part - RP);
  }
  if ((EP == EP_AX || EP == EP_RES || EP == EP_FIN1 || EP == EP_LASTD || kRupd) && a.dot) {
    const int pidx = chunk * tiles + tile;
    block_partial(a.red, a.slot, r, pidx, block_sum_n<NT>(dv.a));
    if (EP == EP_RES) {
      block_partial(a.red, a.slot2, r, pidx, block_sum_n<NT>(dv.b));
      block_partial(a.red, a.slot3, r, pidx, block_sum_n<NT>(dv.c));
    }
  }
}

// Workgroups of the fine operator resident on the device at once for an
// element size and tile: the occupancy of a representative variant (a
// Chebyshev step) times the CU count, looked up once per process.  (The
// variants with a grid transfer hold more LDS, so fewer of theirs may be: a
// chunk length that gives the others one round can give them two.)
template <typename T, int TJ, int TK>
static int tiled_resident_of() {
  int per_cu = 0, dev = 0, cus = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_tiled<T, ST_PLAIN, EP_STEP, TJ, TK, false>, TJ * TK, 0) !=
          hipSuccess ||
      hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || per_cu < 1 ||
      cus < 1)
    throw std::runtime_error("occupancy query of the fine operator failed");
  return per_cu * cus;
}

static int tiled_resident(int sz, const TileShape &ts) {
  static std::atomic<int> cache[2][kNumTileShapes] = {};
  const int v = (ts.tj == 8 && ts.tk == 32) ? 2 : (ts.tj == 16 && ts.tk == 32) ? 3 : 1, d = sz == 8 ? 1 : 0;
  int r = cache[d][v].load(std::memory_order_relaxed);
  if (r > 0) return r;
  if (d == 0)
    r = v == 2 ? tiled_resident_of<float, 8, 32>() : v == 3 ? tiled_resident_of<float, 16, 32>()
                                                           : tiled_resident_of<float, 16, 16>();
  else
    r = v == 2 ? tiled_resident_of<double, 8, 32>() : v == 3 ? tiled_resident_of<double, 16, 32>()
                                                            : tiled_resident_of<double, 16, 16>();
  cache[d][v].store(r, std::memory_order_relaxed);
  return r;
}

template <typename T, int ST, int EP, int TJ, int TK>
static void tiled_go(const Dims &g, int R, const T *E, const ModeC<T> &mc, const OpArgs<T> &a,
                     hipStream_t s, int shape, hipEvent_t ev0, hipEvent_t ev1) {
  const int tiles_k = (g.nz + TK - 1) / TK, tiles_j = (g.ny + TJ - 1) / TJ;
  constexpr bool fused = EP == EP_PRE || ST == ST_PROLONG || ST == ST_DPROLONG;
  const int TI = tiled_chunk(g, R, shape, (int)sizeof(T), fused);
  const int tiles = tiles_j * tiles_k, chunks = (g.nx + TI - 1) / TI;
  // non-temporal output stores once one output vector (all right-hand
  // sides) passes 128 MiB: 64^3 x 16 cells (302 MB in FP32) gains 1-2% from
  // them; 48^3 x 16 cells (127 MB) loses, since the next launch finds such a
  // vector still in the 256 MB last-level cache (one 64^3 cell in FP64, 38
  // MB, solves as fast either way)
  OpArgs<T> an = a;
  an.spread = spread_rule(a.spread, tiles * chunks, kSpreadFine, g.nx % TI == 0);
  an.nt = (size_t)R * 3 * (size_t)g.V * sizeof(T) >= ((size_t)128 << 20) ? 1 : 0;
  if (R % kRHS) throw std::runtime_error("right-hand sides must come in groups of six");
  if (fused &&
      (a.gc.nx * 2 != g.nx || a.gc.ny * 2 != g.ny || a.gc.nz * 2 != g.nz || (TI & 1)))
    throw std::runtime_error("fused grid transfers need the halved grid and chunks of even length");
  // buffer resources address a right-hand side's vector with 32-bit offsets
  if ((size_t)3 * g.V * sizeof(T) >= ((size_t)1 << 31)) throw std::runtime_error("grid too large for the tiled operator");
  const int grid = tiles * chunks * (EP == EP_AXD ? R / kRHS : R);
  if (ev0) {
    // timed launch: the runtime records the events at the kernel's own start
    // and end, so no queue gap is counted
    hipExtLaunchKernelGGL((k_tiled<T, ST, EP, TJ, TK, EP == EP_PRE>), dim3(grid), dim3(TJ * TK), 0, s, ev0, ev1,
                          0, g, E, mc, an, TI, tiles_k, tiles, chunks);
    return;
  }
  hipLaunchKernelGGL((k_tiled<T, ST, EP, TJ, TK, EP == EP_PRE>), dim3(grid), dim3(TJ * TK), 0, s, g, E, mc, an,
                     TI, tiles_k, tiles, chunks);
}

template <typename T, int ST, int EP>
static void tiled_shape(const Dims &g, int R, const T *E, const ModeC<T> &mc, const OpArgs<T> &a, hipStream_t s,
                        int shape, hipEvent_t ev0, hipEvent_t ev1) {
  const TileShape ts = tile_of(g, R, shape);
  if (ts.tj == 8 && ts.tk == 32)
    tiled_go<T, ST, EP, 8, 32>(g, R, E, mc, a, s, shape, ev0, ev1);
  else if (ts.tj == 16 && ts.tk == 32)
    tiled_go<T, ST, EP, 16, 32>(g, R, E, mc, a, s, shape, ev0, ev1);
  else
    tiled_go<T, ST, EP, 16, 16>(g, R, E, mc, a, s, shape, ev0, ev1);
}

template <typename T>
void launch_tiled(int st, int ep, const Dims &g, int R, const T *E, const ModeCoef &m,
                  const OpArgs<T> &a, hipStream_t s, int shape, hipEvent_t ev0, hipEvent_t ev1) {
  // the 9 distinct coefficients, checked against every entry of the table
  ModeC<T> mc;
  double dv[5] = {0, 0, 0, 0, 0}, xv[4] = {0, 0, 0, 0};
  for (int c = 0; c < 3; c++)
    for (int sm = 1; sm < 8; sm++) {
      dv[mode_diag_index(c, sm)] = m.diag[c][sm];
      for (int d = 0; d < 3; d++)
        if (d != c && mode_bit(sm, c) != mode_bit(sm, d)) xv[mode_cross_index(c, d, sm)] = m.cross[c][d][sm];
    }
  for (int c = 0; c < 3; c++)
    for (int sm = 1; sm < 8; sm++) {
      double err = std::fabs(dv[mode_diag_index(c, sm)] - m.diag[c][sm]);
      for (int d = 0; d < 3; d++)
        if (d != c && mode_bit(sm, c) != mode_bit(sm, d))
          err = std::fmax(err, std::fabs(xv[mode_cross_index(c, d, sm)] - m.cross[c][d][sm]));
        else if (d != c && m.cross[c][d][sm] != 0.0)
          err = 1.0;
      if (err > 1e-15 * std::fabs(dv[2])) throw std::runtime_error("mode coupling is not cube-symmetric");
    }
  for (int q = 0; q < 5; q++) mc.d[q] = (T)dv[q];
  for (int q = 0; q < 4; q++) mc.x[q] = (T)xv[q];
#define GO(S_, E_)                                     \
  if (st == S_ && ep == E_) {                          \
    tiled_shape<T, S_, E_>(g, R, E, mc, a, s, shape, ev0, ev1);  \
    return;                                            \
  }
  GO(ST_PLAIN, EP_AX)
  GO(ST_PLAIN, EP_AXD)
  GO(ST_PUPD, EP_AX)
  GO(ST_PLAIN, EP_RES)
  GO(ST_PLAIN, EP_PRE)
  GO(ST_DSCALE, EP_PRE)
  GO(ST_DSCALE, EP_STEP)
  GO(ST_DSCALE, EP_LAST)
  GO(ST_PLAIN, EP_STEP)
  GO(ST_PLAIN, EP_LAST)
  GO(ST_PLAIN, EP_LASTD)
  GO(ST_PROLONG, EP_CHEB0)
  GO(ST_PROLONG, EP_FIN1)
  GO(ST_DPROLONG, EP_CHEB0)
  GO(ST_DPROLONG, EP_FIN1)
  if constexpr (sizeof(T) == 4) {
    GO(ST_PUPDX, EP_AX)
    GO(ST_RUPD, EP_PRE)
  }
#undef GO
  throw std::runtime_error("no operator kernel for this stage/epilogue pair");
}

// ---------------------------------------------------------------------------
// coarse levels: 27-point block stencils, every active RHS per thread (the
// nine coefficients of a block are loaded once for all load cases)
template <typename T, int ST>
__device__ __forceinline__ T stage_at(const OpArgs<T> &a, const T *__restrict__ Ds, T ti, size_t off,
                                      int V, int c, int n) {
  T v = a.u[off + (size_t)c * V + n];
  if (ST == ST_DSCALE) v *= ti * Ds[(size_t)c * V + n];
  return v;
}

// Stencil block `off` of node n (stencil_index layout); `tr`: as the
// transposed block seen from the neighbour, S(m, o) = S(m + o, 26 - o)^T
// (the Galerkin operator is symmetric)
template <typename T>
__device__ __forceinline__ void load_block(const T *__restrict__ Ss, int off, int V, int n, bool tr, T (&sv)[9]) {
  T w[9];
#pragma unroll
  for (int q = 0; q < 9; q++) w[q] = Ss[stencil_index(off, q, V, n)];
#pragma unroll
  for (int c = 0; c < 3; c++)
#pragma unroll
    for (int d = 0; d < 3; d++) sv[3 * c + d] = tr ? w[3 * d + c] : w[3 * c + d];
}

// Coarse-level node update for NR right-hand sides of one sample (load cases
// lc0 .. lc0+NR-1, those set in `mask`): the 27 3x3 blocks of the node's
// stencil row are read once and applied to every right-hand side.  With
// `sym` the 13 lower-offset blocks are taken as the transposed upper blocks
// of the neighbours, S(n, o)[c][d] = S(n + o, -o)[d][c] (the Galerkin
// operator is symmetric), so only 14 of the 27 stored blocks are read; a
// level with a dimension of 2 (where n + o = n - o) reads all 27.
template <typename T, int ST, int EP, int NR>
__device__ __forceinline__ void stencil_node(const Dims &g, const T *__restrict__ S, const OpArgs<T> &a,
                                             int n, int smp, int lc0, unsigned mask, bool sym) {
  int i, j, k;
  node_ijk(g, n, i, j, k);
  const int I[3] = {i == 0 ? g.nx - 1 : i - 1, i, i == g.nx - 1 ? 0 : i + 1};
  const int J[3] = {j == 0 ? g.ny - 1 : j - 1, j, j == g.ny - 1 ? 0 : j + 1};
  const int K[3] = {k == 0 ? g.nz - 1 : k - 1, k, k == g.nz - 1 ? 0 : k + 1};
  const int V = g.V;
  const T *__restrict__ Ss = S + (size_t)smp * 243 * V;
  const T *__restrict__ Ds = a.Dinv ? a.Dinv + (size_t)smp * 3 * V : nullptr;
  const T ti = a.cheb ? (T)a.cheb[smp] : (T)0;
  const T c1 = a.cheb ? (T)a.cheb[kMaxB + smp] : (T)0, c2 = a.cheb ? (T)a.cheb[2 * kMaxB + smp] : (T)0;
  const size_t off0 = (size_t)(smp * kRHS + lc0) * 3 * V;
  T acc[NR][3];
#pragma unroll
  for (int t = 0; t < NR; t++) acc[t][0] = acc[t][1] = acc[t][2] = 0;
#pragma unroll 3
  for (int o = 0; o < 27; o++) {
    const int nb = (I[o / 9] * g.ny + J[(o / 3) % 3]) * g.nz + K[o % 3];
    T sv[9];
    if (sym && o < 13)
      load_block(Ss, 26 - o, V, nb, true, sv);
    else
      load_block(Ss, o, V, n, false, sv);
#pragma unroll
    for (int t = 0; t < NR; t++) {
      if (!((mask >> t) & 1u)) continue;
      const size_t off = off0 + (size_t)t * 3 * V;
      const T u0 = stage_at<T, ST>(a, Ds, ti, off, V, 0, nb), u1 = stage_at<T, ST>(a, Ds, ti, off, V, 1, nb),
              u2 = stage_at<T, ST>(a, Ds, ti, off, V, 2, nb);
      acc[t][0] += sv[0] * u0 + sv[1] * u1 + sv[2] * u2;
      acc[t][1] += sv[3] * u0 + sv[4] * u1 + sv[5] * u2;
      acc[t][2] += sv[6] * u0 + sv[7] * u1 + sv[8] * u2;
    }
  }
#pragma unroll
  for (int t = 0; t < NR; t++) {
    if (!((mask >> t) & 1u)) continue;
    const size_t off = off0 + (size_t)t * 3 * V;
    T uo[3];
#pragma unroll
    for (int c = 0; c < 3; c++) uo[c] = stage_at<T, ST>(a, Ds, ti, off, V, c, n);
    DotAcc dv;
    EpiIn<T> pin;
    epi_load<T, ST, EP>(a, Ds, off, V, n, pin);
    epilogue<T, ST, EP>(a, pin, ti, c1, c2, off, V, n, acc[t], uo, dv);
  }
}

// All load cases of a sample per thread (blockIdx.y = sample), reading the
// stencil once; the small levels run k_stencil_split below.
template <typename T, int ST, int EP>
__global__ __launch_bounds__(kBlock) void k_stencil(Dims g, const T *__restrict__ S, OpArgs<T> a,
                                                    int sym) {
  const int smp = blockIdx.y;
  unsigned mask = 0;
#pragma unroll
  for (int t = 0; t < kRHS; t++) mask |= a.act[smp * kRHS + t] ? (1u << t) : 0u;
  if (!mask) return;
  for (int n = blockIdx.x * kBlock + threadIdx.x; n < g.V; n += gridDim.x * kBlock)
    stencil_node<T, ST, EP, kRHS>(g, S, a, n, smp, 0, mask, sym != 0);
}

// Small levels (a few thousand nodes: too few threads to cover the latency of
// a node's 27 dependent block loads): NR right-hand sides per workgroup row
// (blockIdx.y) and 64 consecutive nodes per workgroup, whose stencil rows are
// split over nine waves -- wave w = 3 di + dj applies the three blocks
// (di, dj, 0..2) -- so a thread's load chain is three blocks long.  The nine
// partial sums meet in LDS and wave t finishes the nodes of right-hand side t.
// Same block order and symmetric reads as stencil_node; only the summation
// order differs.
constexpr int kSplitNodes = 64, kSplitWaves = 9;

template <typename T, int ST, int EP, int NR>
__global__ __launch_bounds__(kSplitNodes *kSplitWaves) void k_stencil_split(Dims g, const T *__restrict__ S,
                                                                             OpArgs<T> a, int sym) {
  const int r0 = EP == EP_AXD ? (int)blockIdx.y * kRHS : (int)blockIdx.y * NR;
  unsigned mask = 0;
#pragma unroll
  for (int t = 0; t < NR; t++) mask |= a.act[r0 + t] ? (1u << t) : 0u;
  if (!mask) return;
  const int smp = r0 / kRHS, lane = threadIdx.x % kSplitNodes, w = threadIdx.x / kSplitNodes;
  const int n = blockIdx.x * kSplitNodes + lane;
  const bool live = n < g.V;
  const int V = g.V;
  const T *__restrict__ Ss = S + (size_t)smp * 243 * V;
  const T *__restrict__ Ds = a.Dinv ? a.Dinv + (size_t)smp * 3 * V : nullptr;
  const T ti = a.cheb ? (T)a.cheb[smp] : (T)0;
  const size_t off0 = (size_t)r0 * 3 * V, offw = off0 + (size_t)w * 3 * V;
  __shared__ T part[NR][kSplitWaves][3][kSplitNodes];
  T acc[NR][3];
#pragma unroll
  for (int t = 0; t < NR; t++) acc[t][0] = acc[t][1] = acc[t][2] = 0;
  // (wave t finishes right-hand side t: what its epilogue reads is asked for
  // first, so that it arrives with the stencil row and not after it)
  const bool fin = w < NR && live && ((mask >> w) & 1u);
  EpiIn<T> pin;
  T uo[3];
  if (fin) {
    epi_load<T, ST, EP>(a, Ds, offw, V, n, pin);
#pragma unroll
    for (int c = 0; c < 3; c++) uo[c] = stage_at<T, ST>(a, Ds, ti, offw, V, c, n);
  }
  if (live) {
    int i, j, k;
    node_ijk(g, n, i, j, k);
    const int di = w / 3, dj = w % 3;
    const int row = (wrap1(i - 1 + di, g.nx) * g.ny + wrap1(j - 1 + dj, g.ny)) * g.nz;
    const int K[3] = {wrap1(k - 1, g.nz), k, wrap1(k + 1, g.nz)};
#pragma unroll
    for (int dk = 0; dk < 3; dk++) {
      const int o = 3 * w + dk, nb = row + K[dk];
      T sv[9];
      if (sym && o < 13)
        load_block(Ss, 26 - o, V, nb, true, sv);
      else
        load_block(Ss, o, V, n, false, sv);
#pragma unroll
      for (int t = 0; t < NR; t++) {
        if (NR > 1 && !((mask >> t) & 1u)) continue;
        const size_t off = off0 + (size_t)t * 3 * V;
        const T u0 = stage_at<T, ST>(a, Ds, ti, off, V, 0, nb), u1 = stage_at<T, ST>(a, Ds, ti, off, V, 1, nb),
                u2 = stage_at<T, ST>(a, Ds, ti, off, V, 2, nb);
        acc[t][0] += sv[0] * u0 + sv[1] * u1 + sv[2] * u2;
        acc[t][1] += sv[3] * u0 + sv[4] * u1 + sv[5] * u2;
        acc[t][2] += sv[6] * u0 + sv[7] * u1 + sv[8] * u2;
      }
    }
  }
#pragma unroll
  for (int t = 0; t < NR; t++)
#pragma unroll
    for (int c = 0; c < 3; c++) part[t][w][c][lane] = acc[t][c];
  __syncthreads();
  if (!fin) return;
  T Au[3];
#pragma unroll
  for (int c = 0; c < 3; c++) {
    T s = part[w][0][c][lane];
#pragma unroll
    for (int q = 1; q < kSplitWaves; q++) s += part[w][q][c][lane];
    Au[c] = s;
  }
  const T c1 = a.cheb ? (T)a.cheb[kMaxB + smp] : (T)0, c2 = a.cheb ? (T)a.cheb[2 * kMaxB + smp] : (T)0;
  DotAcc dv;
  epilogue<T, ST, EP>(a, pin, ti, c1, c2, offw, V, n, Au, uo, dv);
}

// One-plane form of the tiled stencil kernel, for levels with planes of at
// least one 16x16 tile.  A workgroup owns one node plane i of a 16x16 (j,k)
// tile and NG load cases of one sample.  The staged neighbour planes i-1, i,
// i+1 (with the one-node j/k halo, as stage_at stages them) pass through a
// two-buffer LDS ring in three phases -- plane i+1 is loaded into registers
// while plane i-1 is used, and written over it after a barrier -- and each
// phase applies the nine 3x3 blocks of the node's stencil row that couple
// to that plane.  Against a three-plane ring this needs 2/3 of the LDS, so
// more workgroups share a CU and hide the coefficient loads' latency.

// Stencil coefficients through a raw buffer resource (bload): a scalar block
// offset plus one 32-bit lane offset per load (no vector address
// arithmetic), a node's block as two 16-byte loads and one scalar load
// (stencil_index layout), and a load past the sample's stencil returns 0
// instead of faulting.

constexpr int kStBatch = 3;  // stencil blocks whose coefficient loads are issued together

template <typename T, int ST, int EP, int NG, int SYM>
__global__ __launch_bounds__(kBlock) void k_stencil_plane(Dims g, const T *__restrict__ S, OpArgs<T> a,
                                                          int tiles_k, int tiles) {
  constexpr int G = EP == EP_AXD ? 1 : kRHS / NG;  // load-case groups per sample
  // units of (plane, tile), the groups of a unit next to each other
  const WorkId id = work_order(blockIdx.x, gridDim.x, gridDim.x / (G * tiles * g.nx), tiles * g.nx, G, a.spread);
  const int tile = id.unit % tiles, i = id.unit / tiles;
  const int smp = id.cell, lc0 = id.inner * NG;
  unsigned mask = 0;
#pragma unroll
  for (int t = 0; t < NG; t++) mask |= a.act[smp * kRHS + lc0 + t] ? (1u << t) : 0u;
  if (!mask) return;
  __shared__ T us[2][NG][3][kTN * kTN];
  const int tid = threadIdx.x;
  const int j0 = (tile / tiles_k) * kTile, k0 = (tile % tiles_k) * kTile;
  const int V = g.V, plane = g.ny * g.nz;
  constexpr unsigned SZ = sizeof(T);
  const unsigned vb = (unsigned)V * SZ;  // bytes per V stencil values
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      (void *)(S + (size_t)smp * 243 * V), (short)0, (int)(243u * vb), 0x00020000);
  const T *__restrict__ Ds = a.Dinv ? a.Dinv + (size_t)smp * 3 * V : nullptr;
  const T ti = a.cheb ? (T)a.cheb[smp] : (T)0;
  const T c1 = a.cheb ? (T)a.cheb[kMaxB + smp] : (T)0, c2 = a.cheb ? (T)a.cheb[2 * kMaxB + smp] : (T)0;
  const size_t off0 = (size_t)(smp * kRHS + lc0) * 3 * V;
  int soff[2];
#pragma unroll
  for (int q = 0; q < 2; q++) {
    const int t = tid + q * kBlock;
    soff[q] = -1;
    if (t < kTN * kTN) {
      const int nj = t / kTN, nk = t - nj * kTN;
      soff[q] = wrap1(j0 - 1 + nj, g.ny) * g.nz + wrap1(k0 - 1 + nk, g.nz);
    }
  }
  T stg[2][NG][3];
  auto fetch = [&](int ip) {
    const int iw = wrap1(ip, g.nx);
#pragma unroll
    for (int q = 0; q < 2; q++) {
      if (soff[q] < 0) continue;
      const int n = iw * plane + soff[q];
      // the sample's inverse diagonal is shared by its load cases
      T sc[3] = {1, 1, 1};
      if (ST == ST_DSCALE) {
#pragma unroll
        for (int c = 0; c < 3; c++) sc[c] = ti * Ds[(size_t)c * V + n];
      }
#pragma unroll
      for (int r = 0; r < NG; r++)
        // inactive load cases stage zeros: the phases then run branch-free
#pragma unroll
        for (int c = 0; c < 3; c++)
          stg[q][r][c] = ((mask >> r) & 1u) ? a.u[off0 + (size_t)r * 3 * V + (size_t)c * V + n] * sc[c] : (T)0;
    }
  };
  auto put = [&](int buf) {
#pragma unroll
    for (int q = 0; q < 2; q++) {
      if (soff[q] < 0) continue;
      const int t = tid + q * kBlock;
#pragma unroll
      for (int r = 0; r < NG; r++)
#pragma unroll
        for (int c = 0; c < 3; c++) us[buf][r][c][t] = stg[q][r][c];
    }
  };
  const int nj = tid / kTile, nk = tid % kTile;
  const int gj = j0 + nj, gk = k0 + nk;
  const bool owns = gj < g.ny && gk < g.nz;
  const int Jn[3] = {wrap1(gj - 1, g.ny), wrap1(gj, g.ny), wrap1(gj + 1, g.ny)};
  const int Kn[3] = {wrap1(gk - 1, g.nz), wrap1(gk, g.nz), wrap1(gk + 1, g.nz)};
  const int n = i * plane + gj * g.nz + gk;
  T acc[NG][3];
#pragma unroll
  for (int t = 0; t < NG; t++) acc[t][0] = acc[t][1] = acc[t][2] = 0;
  // the nine blocks of offset plane di (0: i-1, 1: i, 2: i+1) against the
  // staged plane in buffer `buf`
  auto phase = [&](int di, int buf) {
    const int pw = wrap1(i - 1 + di, g.nx);
#pragma unroll
    for (int pos = 0; pos < 9; pos++) {
      const int dj = pos / 3, dk = pos % 3;
      const int o = di * 9 + pos;
      const int slot = (nj + dj) * kTN + nk + dk;
      T sv[9];
      {
        // S(n, o) = S(n + o, 26 - o)^T for the lower offsets
        const bool tr = SYM && o < 13;
        const int ob = tr ? 26 - o : o;
        const unsigned node = tr ? (unsigned)(pw * plane + Jn[dj] * g.nz + Kn[dk]) : (unsigned)n;
        const unsigned base = (unsigned)(ob * 9) * vb;  // block ob (stencil_index layout)
        // (the four consecutive loads of each [V][4] group are issued by
        // the compiler as one 16-byte load)
        T w[9];
#pragma unroll
        for (int q = 0; q < 4; q++) {
          w[q] = bload(rs, (node * 4u + q) * SZ, base, (T *)nullptr);
          w[4 + q] = bload(rs, (node * 4u + q) * SZ, base + 4u * vb, (T *)nullptr);
        }
        w[8] = bload(rs, node * SZ, base + 8u * vb, (T *)nullptr);
#pragma unroll
        for (int c = 0; c < 3; c++)
#pragma unroll
          for (int d = 0; d < 3; d++) sv[3 * c + d] = tr ? w[3 * d + c] : w[3 * c + d];
      }
#pragma unroll
      for (int t = 0; t < NG; t++) {
        const T u0 = us[buf][t][0][slot], u1 = us[buf][t][1][slot], u2 = us[buf][t][2][slot];
#pragma unroll
        for (int c = 0; c < 3; c++) {
          T v = acc[t][c];
          v = fma(sv[3 * c], u0, v);
          v = fma(sv[3 * c + 1], u1, v);
          acc[t][c] = fma(sv[3 * c + 2], u2, v);
        }
      }
      // coefficient loads are issued kStBatch blocks at a time: the sums are
      // pinned here, so the compiler neither sinks the FMAs into the
      // epilogue nor hoists all 81 loads of the phase ahead of them (which
      // costs occupancy)
      if (pos % kStBatch == kStBatch - 1) {
#pragma unroll
        for (int t = 0; t < NG; t++)
#pragma unroll
          for (int c = 0; c < 3; c++) asm volatile("" : "+v"(acc[t][c]));
      }
    }
  };
  fetch(i - 1);
  put(0);
  fetch(i);
  put(1);
  fetch(i + 1);  // in flight during the first phase
  __syncthreads();
  if (owns) phase(0, 0);
  __syncthreads();
  put(0);
  T uo[NG][3];
  if (owns) {
    phase(1, 1);
#pragma unroll
    for (int t = 0; t < NG; t++)
#pragma unroll
      for (int c = 0; c < 3; c++) uo[t][c] = us[1][t][c][(nj + 1) * kTN + nk + 1];
  }
  __syncthreads();
  if (owns) {
    phase(2, 0);
#pragma unroll
    for (int t = 0; t < NG; t++) {
      if (!((mask >> t) & 1u)) continue;
      const size_t off = off0 + (size_t)t * 3 * V;
      DotAcc dv;
      EpiIn<T> pin;
      epi_load<T, ST, EP>(a, Ds, off, V, n, pin);
      epilogue<T, ST, EP>(a, pin, ti, c1, c2, off, V, n, acc[t], uo[t], dv);
    }
  }
}

template <typename T>
void launch_stencil(int st, int ep, const Dims &g, int R, const T *S, const OpArgs<T> &a,
                    hipStream_t s, int cells) {
  const int blocks = (g.V + kBlock - 1) / kBlock;
  const int nsmp = (R + kRHS - 1) / kRHS;
  const int sym = (g.nx > 2 && g.ny > 2 && g.nz > 2) ? 1 : 0;
  // planes of at least one full 16x16 tile: the one-plane LDS kernel (all six
  // load cases of a sample per workgroup in FP32, 47 KB of LDS: the stencil
  // row is read once per node; three in FP64), once that gives a workgroup
  // per CU.  One cell, and FP64 in general, take it with three load cases per
  // workgroup from 192 workgroups on: the nine-wave split kernel below re-reads
  // the row for every load case (a smoothing step of one cell: FP32 32^3, 17.3
  // -> 9.7 us; FP64 30 x 22 x 26, 240 workgroups, 30.8 -> 13.6 us).  Around that
  // line, whole solves of one cell with 16-wide levels, split -> one-plane, FP64
  // and mixed: 96 workgroups 8.9 -> 9.2 and 4.1 -> 4.3 ms, 128 9.3 -> 9.1 and
  // 3.85 -> 3.91 (with 32 x 16 planes 8.5 -> 8.7 and 3.5 -> 3.65), 160 11.0 ->
  // 10.2 and 4.3 -> 4.2, 192 13.7 -> 12.2 and 5.0 -> 4.8, 256 17.5 -> 14.9 and
  // 6.0 -> 5.4.  The power iteration runs one load case.
  const int tiles_k = (g.nz + kTile - 1) / kTile, tiles_j = (g.ny + kTile - 1) / kTile;
  const long units = (long)tiles_j * tiles_k * g.nx;
  // (and a sample's stencil addressable by a buffer resource: < 2 GiB)
  const bool fits = g.ny >= kTile && g.nz >= kTile && g.nx >= 3 && R % kRHS == 0 &&
                    (size_t)243 * g.V * sizeof(T) < ((size_t)1 << 31);
  int ng = 0;  // load cases per workgroup of the one-plane kernel (0: not taken)
  if (fits && sizeof(T) == 4 && units * cells >= 256)
    ng = kRHS;
  else if (fits && (sizeof(T) == 8 || nsmp == 1) && units * cells * 2 >= 192)
    ng = kRHS / 2;
  const unsigned pl_blocks = ng ? (unsigned)(units * nsmp * (kRHS / ng)) : 0u;
  // all load cases per thread once that still leaves >= 2 workgroups per CU
  const bool multi = (long)blocks * cells >= 512 && R % kRHS == 0;
  const int split_blocks = (g.V + kSplitNodes - 1) / kSplitNodes;
  // two right-hand sides per split workgroup once one each gives a workgroup
  // per CU: they share the stencil row, which every right-hand side otherwise
  // reads from L2 again (16^3, one cell in FP64, 384 workgroups: 7.0 -> 5.7 us a
  // step; three per workgroup, 128 left: 6.6 us)
  const int nr = R % kRHS == 0 && (long)split_blocks * cells * kRHS >= 256 ? 2 : 1;
  OpArgs<T> an = a;
  an.spread = spread_rule(a.spread, (int)units, kSpreadStencil, true);
#define PLANE(S_, E_, NG_, SYM_, GRID_)                                                             \
  hipLaunchKernelGGL((k_stencil_plane<T, S_, E_, NG_, SYM_>), dim3(GRID_), dim3(kBlock), 0, s, g, S, an, tiles_k, \
                     tiles_j *tiles_k)
#define GO(S_, E_)                                                                               \
  if (st == S_ && ep == E_) {                                                                    \
    if constexpr (E_ == EP_AXD) {                                                                \
      if (ng && sym) PLANE(S_, E_, 1, 1, (unsigned)(units * nsmp));                              \
      else if (ng) PLANE(S_, E_, 1, 0, (unsigned)(units * nsmp));                                \
    } else {                                                                                     \
      if constexpr (sizeof(T) == 4) {                                                            \
        if (ng == kRHS && sym) PLANE(S_, E_, kRHS, 1, pl_blocks);                                \
        else if (ng == kRHS) PLANE(S_, E_, kRHS, 0, pl_blocks);                                  \
      }                                                                                          \
      if (ng == kRHS / 2 && sym) PLANE(S_, E_, kRHS / 2, 1, pl_blocks);                          \
      else if (ng == kRHS / 2) PLANE(S_, E_, kRHS / 2, 0, pl_blocks);                            \
    }                                                                                            \
    if (ng) return;                                                                              \
    if (multi)                                                                                   \
      hipLaunchKernelGGL((k_stencil<T, S_, E_>), dim3(blocks, nsmp), dim3(kBlock), 0, s, g, S,       \
                         a, sym);                                                                \
    else if (E_ == EP_AXD || nr == 1)                                                            \
      hipLaunchKernelGGL((k_stencil_split<T, S_, E_, 1>), dim3(split_blocks, E_ == EP_AXD ? nsmp : R), \
                         dim3(kSplitNodes * kSplitWaves), 0, s, g, S, a, sym);                   \
    else                                                                                         \
      hipLaunchKernelGGL((k_stencil_split<T, S_, E_, 2>), dim3(split_blocks, R / 2),             \
                         dim3(kSplitNodes * kSplitWaves), 0, s, g, S, a, sym);                   \
    return;                                                                                      \
  }
  GO(ST_PLAIN, EP_AX)
  GO(ST_PLAIN, EP_AXD)
  GO(ST_PLAIN, EP_PRE)
  GO(ST_DSCALE, EP_CHEB0L)
  GO(ST_DSCALE, EP_STEP)
  GO(ST_DSCALE, EP_LAST)
  GO(ST_PLAIN, EP_STEP)
  GO(ST_PLAIN, EP_LAST)
  GO(ST_PLAIN, EP_CHEB0)
  GO(ST_PLAIN, EP_FIN1)
#undef GO
#undef PLANE
  throw std::runtime_error("no operator kernel for this stage/epilogue pair");
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_add2(int V, const T *__restrict__ xn,
                                                 const T *__restrict__ d, T *__restrict__ x,
                                                 const int *__restrict__ act) {
  const int r = blockIdx.y;
  if (!act[r]) return;
  const size_t off = (size_t)r * 3 * V;
  for (int t = blockIdx.x * kBlock + threadIdx.x; t < 3 * V; t += gridDim.x * kBlock)
    x[off + t] = xn[off + t] + d[off + t];
}

template <typename T>
void launch_add2(int V, int R, const T *xn, const T *d, T *x, const int *act, hipStream_t s) {
  hipLaunchKernelGGL(k_add2<T>, dim3(grid_for(3 * V), R), dim3(kBlock), 0, s, V, xn, d, x, act);
}

#define FEMH_OPS_INST(T)                                                                        \
  template void launch_tiled<T>(int, int, const Dims &, int, const T *, const ModeCoef &,       \
                                const OpArgs<T> &, hipStream_t, int, hipEvent_t, hipEvent_t);   \
  template void launch_stencil<T>(int, int, const Dims &, int, const T *, const OpArgs<T> &,    \
                                  hipStream_t, int);                                            \
  template void launch_add2<T>(int, int, const T *, const T *, T *, const int *, hipStream_t);

FEMH_OPS_INST(double)
FEMH_OPS_INST(float)

}  // namespace femh
