// 2D acoustic variable-density engine (staggered pressure / velocity,
// 4th-order space, C-PML) for a batch of shots: ONE fused launch per time
// step for the forward/replay and one for the adjoint (+ gradient
// correlation).
//
// Reference semantics (paths relative to the reference root):
//   step       src/models/acoustic/backends/shared/acoustic2D_VD_xPU.jl:1-178
//   stencils   src/utils/fdgen.jl:65-161 (order 4, zero outside the array)
//   driver     src/models/acoustic/acou_gradient.jl:97-203
//   correlate  correlate_gradient_xPU.jl:12-21, acoustic2D_VD_xPU.jl:180-198
//
// Fusion.  The forward step is p <- p - m0 div~ v, inject, v <- v - m1 grad~ p.
// The velocity update needs the *new* pressure one cell left / two right of
// each velocity point, so a block recomputes the new pressure on its tile
// plus that cross-shaped halo in LDS (redundant work on a few % of the
// cells, no extra HBM traffic), then updates the velocities of its tile.
// Because neighbouring blocks read the old state around their tiles, the
// state is double buffered by step parity (read parity it-1, write parity
// it), including the C-PML memory variables.  The adjoint step (v first,
// then p) is fused the same way around the old adjoint pressure, and the
// correlation of grad_m0 / grad_m1 with the replayed pressure is done in
// the same launch.
//
// Memory-level parallelism: every global load a thread needs that does not
// depend on LDS (old pressure, material factors, halo cells) is issued
// before the first barrier, so a block has all its HBM requests in flight
// at once.  Tiles are handed to blocks XCD-aware: the hardware deals blocks
// round-robin over the 8 XCDs, and the block -> tile map gives each XCD a
// contiguous run of tiles so the halo rows shared by neighbouring tiles are
// found in that XCD's L2.
//
// Layout: every field is an nx*nz slab per shot with x fastest.  vx has
// nx-1 valid columns and vz nx*(nz-1) valid rows; the extra column/row is
// kept at zero, which is exactly the zero extension of the reference's
// truncated stencils.
#include <algorithm>
#include <cstdlib>

#include "swx_levels.hpp"
#include "swx_internal.hpp"

namespace swx {
namespace {

constexpr int TX = 64;   // tile width (one wavefront)
constexpr int BY = 4;    // thread rows per block
constexpr int NT = TX * BY;

// tile heights per precision (LDS: forward ~29 KB f32 / 30 KB f64)
template <typename T> struct Tiles;
template <> struct Tiles<float> { static constexpr int fwd_max = 32; };
template <> struct Tiles<double> { static constexpr int fwd_max = 32; };

template <typename T>
struct Vd2dArgs {
  int nx, nz, h;
  int nbx, nbz;                  // tiles per shot along x and z
  int ch;                        // rows per block of the z-marching kernel
  int64_t N;
  T idx, idz;
  const T *m0, *m1x, *m1z;
  const T *p_o, *vx_o, *vz_o;   // read parity (shot 0 slab)
  T *p_n, *vx_n, *vz_n;         // write parity
  const T *psx_o; T *psx_n; int64_t spx;
  const T *psz_o; T *psz_n; int64_t spz;
  const T *xix_o; T *xix_n; int64_t sxx;
  const T *xiz_o; T *xiz_n; int64_t sxz;
  const T *cpml; int cstride;
  PointArgsView pt;
  const T *srctf;
  T *traces;                     // forward recording (nullable)
  const T *res;                  // adjoint residuals
  const int *nt_shot;
  int nsh;                       // shots of the batch (pair kernels)
  int sgrp;                      // shots per group of the block order (vd2d_tile_of)
  int it, act_min;
  // pressure history of the segment: slot k holds p^{base+k}
  T *pbuf; int64_t pslot; int smode; int S; int cbase;
  // gradient correlation (adjoint)
  T *g0, *g1x, *g1z; T idt;
};

template <typename T>
__device__ __forceinline__ T d4(T a, T b, T c, T d) {
  // (1/24) a - (9/8) b + (9/8) c - (1/24) d  (fdgen.jl order 4, deriv 1)
  const T c1 = T(1.0 / 24.0), c2 = T(-9.0 / 8.0);
  return c1 * a + c2 * b + (-c2) * c + (-c1) * d;
}

// Base of the history segment a step stores into, or -1.  Forward (smode
// 1): the final segment of the shot, from its last checkpoint floor(nt/S)*S
// on (the buffer of LinearCheckpointer, checkpointers.jl:44-56); replay
// (smode 2): the segment being replayed.
__device__ __forceinline__ int store_base(int smode, int it, int nts, int S, int cbase) {
  if (smode == 1) {
    const int seg0 = (nts / S) * S;
    return it > seg0 ? seg0 : -1;
  }
  if (smode == 2) return cbase;
  return -1;
}

// Block -> tile map giving each XCD a contiguous run of tiles.
__device__ __forceinline__ int xcd_tile(int b, int nb) {
  const int per = nb >> 3;
  if (b >= per * 8) return b;
  return (b & 7) * per + (b >> 3);
}

// Tile (bx, bz) and shot s of block b of a tiles x shots grid.  The shots
// are taken in groups of sgrp (a divisor of the batch): the blocks of one
// tile for the shots of a group follow each other, then the next tile of
// the group, and a group's tiles form one contiguous run.  Consecutive
// blocks land on one XCD (xcd_tile), so the sgrp blocks of a tile read its
// model factors (3 of the 9 values of a forward cell step) from that XCD's
// L2 after the first; sgrp = 1 is the plain shot-after-shot order.  The
// z-neighbour tile of the same shot stays nbx * sgrp blocks back, within
// L2 reach for small groups.
template <typename T>
__device__ __forceinline__ void vd2d_tile_of(const Vd2dArgs<T> &a, int b, int &bx, int &bz, int &s) {
  const int g = a.sgrp;
  const int lo = b % g, t = b / g;
  const int tiles = a.nbx * a.nbz;
  const int tile = t % tiles;
  s = (t / tiles) * g + lo;
  bx = tile % a.nbx;
  bz = tile / a.nbx;
}

// Is tile (I0, J0) of shot s an interior tile of the forward step: every
// cell the tile step reads or updates is inside the grid and outside the
// C-PML strips, and no source (new-pressure rows) or receiver (tile rows)
// lies in its rows?
template <int TZ, typename T>
__device__ __forceinline__ bool vd2d_fwd_is_lean(const Vd2dArgs<T> &a, int s, int I0, int J0) {
  const int nx = a.nx, nz = a.nz, h = a.h;
  if (!(I0 - 3 >= 0 && I0 - 1 > h && I0 + TX + 3 <= nx - 1 && I0 + TX + 1 < nx - h - 1 && J0 - 3 >= 0 &&
        J0 - 1 > h && J0 + TZ + 3 <= nz - 1 && J0 + TZ + 1 < nz - h - 1))
    return false;
  const int *sr = a.pt.srow + (int64_t)s * (a.pt.nrows + 1);
  const int *rr = a.pt.rrow + (int64_t)s * (a.pt.nrows + 1);
  return sr[J0 - 1] == sr[J0 + TZ + 2] && (a.traces == nullptr || rr[J0] == rr[J0 + TZ]);
}

// Forward / replay step of an interior tile (vd2d_fwd_is_lean): the updates
// of vd2d_fwd_kernel, in the same operand order, without per-cell tests, on
// 32-bit offsets from per-shot bases.
// Cross-shaped halo of the new pressure of a forward tile: columns I0-1,
// I0+TX, I0+TX+1 on the tile rows, rows J0-1, J0+TZ, J0+TZ+1 on the tile
// columns; entry k of thread tid, (lx, lz) in s_p coordinates or -1.
template <int TZ>
__device__ __forceinline__ void fwd_halo_cell(int q, int &lx, int &lz) {
  constexpr int HX = 3 * TZ, H = HX + 3 * TX;
  lx = -1;
  lz = -1;
  if (q < HX) {
    const int col = q / TZ;
    lz = 1 + q % TZ;
    lx = col == 0 ? 0 : TX + col;
  } else if (q < H) {
    const int row = (q - HX) / TX;
    lx = 1 + (q - HX) % TX;
    lz = row == 0 ? 0 : TZ + row;
  }
}

// Model factors an interior forward tile reads (the same for every shot):
// m0, m1x, m1z on the thread's R tile cells, m0 on its halo cells.
template <typename T, int TZ>
struct FwdTileModel {
  static constexpr int R = TZ / BY, HR = (3 * TZ + 3 * TX + NT - 1) / NT;
  T m0[R], m1x[R], m1z[R], hm0[HR];
};

template <typename T, int TZ>
__device__ __forceinline__ void vd2d_fwd_lean_model(const Vd2dArgs<T> &a, int I0, int J0, FwdTileModel<T, TZ> &m) {
  constexpr int R = TZ / BY, HR = FwdTileModel<T, TZ>::HR;
  const int nx = a.nx;
  const int tx = threadIdx.x, ty = threadIdx.y, tid = ty * TX + tx;
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int c = (J0 + ty + BY * r) * nx + I0 + tx;
    m.m0[r] = a.m0[c];
    m.m1x[r] = a.m1x[c];
    m.m1z[r] = a.m1z[c];
  }
#pragma unroll
  for (int k = 0; k < HR; k++) {
    int lx, lz;
    fwd_halo_cell<TZ>(tid + k * NT, lx, lz);
    m.hm0[k] = lx >= 0 ? a.m0[(J0 - 1 + lz) * nx + I0 - 1 + lx] : T(0);
  }
}

template <typename T, int TZ>
__device__ __forceinline__ void vd2d_fwd_lean_tile(const Vd2dArgs<T> &a, int s, int nts, int I0, int J0,
                                                   T (&s_vx)[TZ + 3][TX + 6], T (&s_vz)[TZ + 6][TX + 3],
                                                   T (&s_p)[TZ + 3][TX + 3], const FwdTileModel<T, TZ> &m) {
  constexpr int R = TZ / BY;
  const int nx = a.nx;
  const int tx = threadIdx.x, ty = threadIdx.y, tid = ty * TX + tx;
  const int64_t so = (int64_t)s * a.N;
  const T *__restrict__ po = a.p_o + so;
  const T *__restrict__ vxo = a.vx_o + so;
  const T *__restrict__ vzo = a.vz_o + so;
  // every global load of the thread is issued before its first LDS store
  constexpr int KX = (TZ + 3 + BY - 1) / BY, KZ = (TZ + 6 + BY - 1) / BY;
  T lx0[KX], lx1[KX], lz0[KZ], lz1[KZ];
#pragma unroll
  for (int k = 0; k < KX; k++) {
    const int lz = ty + k * BY;
    const int c = (J0 - 1 + lz) * nx + I0 - 3 + tx;
    lx0[k] = lz < TZ + 3 ? vxo[c] : T(0);
    lx1[k] = lz < TZ + 3 && tx < 6 ? vxo[c + TX] : T(0);
  }
#pragma unroll
  for (int k = 0; k < KZ; k++) {
    const int lz = ty + k * BY;
    const int c = (J0 - 3 + lz) * nx + I0 - 1 + tx;
    lz0[k] = lz < TZ + 6 ? vzo[c] : T(0);
    lz1[k] = lz < TZ + 6 && tx < 3 ? vzo[c + TX] : T(0);
  }
  T rp[R];
#pragma unroll
  for (int r = 0; r < R; r++) rp[r] = po[(J0 + ty + BY * r) * nx + I0 + tx];
  constexpr int HR = FwdTileModel<T, TZ>::HR;
  T hp[HR];
  int hlx[HR], hlz[HR];
#pragma unroll
  for (int k = 0; k < HR; k++) {
    fwd_halo_cell<TZ>(tid + k * NT, hlx[k], hlz[k]);
    hp[k] = hlx[k] >= 0 ? po[(J0 - 1 + hlz[k]) * nx + I0 - 1 + hlx[k]] : T(0);
  }
  const T(&rm0)[R] = m.m0;
  const T(&rm1x)[R] = m.m1x;
  const T(&rm1z)[R] = m.m1z;
  const T(&hm0)[HR] = m.hm0;
#pragma unroll
  for (int k = 0; k < KX; k++) {
    const int lz = ty + k * BY;
    if (lz < TZ + 3) {
      s_vx[lz][tx] = lx0[k];
      if (tx < 6) s_vx[lz][TX + tx] = lx1[k];
    }
  }
#pragma unroll
  for (int k = 0; k < KZ; k++) {
    const int lz = ty + k * BY;
    if (lz < TZ + 6) {
      s_vz[lz][tx] = lz0[k];
      if (tx < 3) s_vz[lz][TX + tx] = lz1[k];
    }
  }
  __syncthreads();
  const int sb = store_base(a.smode, a.it, nts, a.S, a.cbase);
  T *__restrict__ pn = a.p_n + so;
  auto lean_p = [&](int lx, int lz, T pold, T m0v) -> T {
    const T dvx = d4(s_vx[lz][lx], s_vx[lz][lx + 1], s_vx[lz][lx + 2], s_vx[lz][lx + 3]) * a.idx;
    const T dvz = d4(s_vz[lz][lx], s_vz[lz + 1][lx], s_vz[lz + 2][lx], s_vz[lz + 3][lx]) * a.idz;
    return pold - m0v * (dvx + dvz);
  };
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int lz = ty + BY * r + 1;
    const T pv = lean_p(tx + 1, lz, rp[r], rm0[r]);
    s_p[lz][tx + 1] = pv;
    const int c = (J0 + lz - 1) * nx + I0 + tx;
    st_nt(pn + c, pv);
    if (sb >= 0) {
      T *hs = a.pbuf + so;
      st_nt(hs + (int64_t)(a.it - sb) * a.pslot + c, pv);
      if (a.smode == 1 && a.it == sb + 1) st_nt(hs + c, rp[r]);
    }
  }
#pragma unroll
  for (int k = 0; k < HR; k++)
    if (hlx[k] >= 0) s_p[hlz[k]][hlx[k]] = lean_p(hlx[k], hlz[k], hp[k], hm0[k]);
  __syncthreads();
  T *__restrict__ vxn = a.vx_n + so;
  T *__restrict__ vzn = a.vz_n + so;
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int lz = ty + BY * r;
    const int c = (J0 + lz) * nx + I0 + tx;
    const T dx = d4(s_p[lz + 1][tx], s_p[lz + 1][tx + 1], s_p[lz + 1][tx + 2], s_p[lz + 1][tx + 3]) * a.idx;
    const T vx = s_vx[lz + 1][tx + 3] - rm1x[r] * dx;
    st_nt(vxn + c, vx);
    const T dz = d4(s_p[lz][tx + 1], s_p[lz + 1][tx + 1], s_p[lz + 2][tx + 1], s_p[lz + 3][tx + 1]) * a.idz;
    const T vz = s_vz[lz + 3][tx + 1] - rm1z[r] * dz;
    st_nt(vzn + c, vz);
  }
}

// Interior tiles of a forward / replay step; blocks of other tiles return at
// once and vd2d_fwd_kernel<T, TZ, false>, launched right after on the same
// grid, steps them.
template <typename T, int TZ>
__global__ __launch_bounds__(NT) void vd2d_fwd_lean(Vd2dArgs<T> a) {
  int bx, bz, s;
  vd2d_tile_of(a, xcd_tile(blockIdx.x, gridDim.x), bx, bz, s);
  const int nts = a.nt_shot[s];
  if (a.it > nts || nts <= a.act_min) return;
  const int I0 = bx * TX, J0 = bz * TZ;
  if (!vd2d_fwd_is_lean<TZ>(a, s, I0, J0)) return;
  __shared__ T s_vx[TZ + 3][TX + 6];
  __shared__ T s_vz[TZ + 6][TX + 3];
  __shared__ T s_p[TZ + 3][TX + 3];
  FwdTileModel<T, TZ> m;
  vd2d_fwd_lean_model<T, TZ>(a, I0, J0, m);
  vd2d_fwd_lean_tile<T, TZ>(a, s, nts, I0, J0, s_vx, s_vz, s_p, m);
}

// Forward / replay step of a tile that is not interior (C-PML strips, grid
// edges, points): update_p_CPML!, injection, recording, then the velocity
// updates with their C-PML memory variables, with per-cell tests.
template <typename T, int TZ>
__device__ __forceinline__ void vd2d_fwd_general_tile(const Vd2dArgs<T> &a, int s, int nts, int I0, int J0,
                                                      T (&s_vx)[TZ + 3][TX + 6], T (&s_vz)[TZ + 6][TX + 3],
                                                      T (&s_p)[TZ + 3][TX + 3], int (&s_pts)[2]) {
  constexpr int R = TZ / BY;
  const int nx = a.nx, nz = a.nz, h = a.h;
  const int tx = threadIdx.x, ty = threadIdx.y, tid = ty * TX + tx;
  const int64_t so = (int64_t)s * a.N;
  const T *cb = a.cpml + (int64_t)s * a.cstride;
  const AxisCoef<T> cx = axis_coef(cb, h, 0), cz = axis_coef(cb, h, 1);

  // ---- phase 0: every load that does not depend on LDS, all issued before
  // the first LDS store -------------------------------------------------------
  constexpr int QX = (TZ + 3) * (TX + 6), KQX = (QX + NT - 1) / NT;
  constexpr int QZ = (TZ + 6) * (TX + 3), KQZ = (QZ + NT - 1) / NT;
  T gvx[KQX], gvz[KQZ];
#pragma unroll
  for (int k = 0; k < KQX; k++) {
    const int q = tid + k * NT;
    const int lz = q / (TX + 6), lx = q % (TX + 6);
    const int gi = I0 - 3 + lx, gj = J0 - 1 + lz;
    T v = 0;
    if (q < QX && gi >= 0 && gi <= nx - 2 && gj >= 0 && gj <= nz - 1) v = a.vx_o[so + (int64_t)gj * nx + gi];
    gvx[k] = v;
  }
#pragma unroll
  for (int k = 0; k < KQZ; k++) {
    const int q = tid + k * NT;
    const int lz = q / (TX + 3), lx = q % (TX + 3);
    const int gi = I0 - 1 + lx, gj = J0 - 3 + lz;
    T v = 0;
    if (q < QZ && gi >= 0 && gi <= nx - 1 && gj >= 0 && gj <= nz - 2) v = a.vz_o[so + (int64_t)gj * nx + gi];
    gvz[k] = v;
  }
  const int gi = I0 + tx;
  T rp[R], rm0[R], rm1x[R], rm1z[R];
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int gj = J0 + ty + BY * r;
    const bool ok = gi < nx && gj < nz;
    const int64_t c = (int64_t)gj * nx + gi;
    rp[r] = ok ? a.p_o[so + c] : T(0);
    rm0[r] = ok ? a.m0[c] : T(0);
    rm1x[r] = ok ? a.m1x[c] : T(0);
    rm1z[r] = ok ? a.m1z[c] : T(0);
  }
  // halo of the new-pressure region: 3 columns x TZ rows, 3 rows x TX columns
  constexpr int HX = 3 * TZ, H = HX + 3 * TX, HR = (H + NT - 1) / NT;
  // does any source lie in the rows whose new pressure this block computes,
  // or any receiver in its tile rows?  (most blocks: no point lookups)
  if (tid == 0) {
    const int *sr = a.pt.srow + (int64_t)s * (a.pt.nrows + 1);
    const int *rr = a.pt.rrow + (int64_t)s * (a.pt.nrows + 1);
    s_pts[0] = sr[max(J0 - 1, 0)] < sr[min(J0 + TZ + 2, nz)];
    s_pts[1] = a.traces != nullptr && rr[J0] < rr[min(J0 + TZ, nz)];
  }
  T hp[HR], hm0[HR];
  int hlx[HR], hlz[HR];
#pragma unroll
  for (int k = 0; k < HR; k++) {
    const int q = tid + k * NT;
    int lx = -1, lz = -1;
    if (q < HX) {
      const int col = q / TZ;
      lz = 1 + q % TZ;
      lx = col == 0 ? 0 : TX + col;
    } else if (q < H) {
      const int row = (q - HX) / TX;
      lx = 1 + (q - HX) % TX;
      lz = row == 0 ? 0 : TZ + row;
    }
    T vp = 0, vm = 0;
    const int gi2 = I0 - 1 + lx, gj2 = J0 - 1 + lz;
    if (lx >= 0 && gi2 >= 0 && gi2 <= nx - 1 && gj2 >= 0 && gj2 <= nz - 1) {
      const int64_t c2 = (int64_t)gj2 * nx + gi2;
      vp = a.p_o[so + c2];
      vm = a.m0[c2];
    }
    hlx[k] = lx;
    hlz[k] = lz;
    hp[k] = vp;
    hm0[k] = vm;
  }
#pragma unroll
  for (int k = 0; k < KQX; k++) {
    const int q = tid + k * NT;
    if (q < QX) s_vx[q / (TX + 6)][q % (TX + 6)] = gvx[k];
  }
#pragma unroll
  for (int k = 0; k < KQZ; k++) {
    const int q = tid + k * NT;
    if (q < QZ) s_vz[q / (TX + 3)][q % (TX + 3)] = gvz[k];
  }
  __syncthreads();

  // ---- phase 1: new pressure (update_p_CPML! + inject_sources!) ----------
  const int sb = store_base(a.smode, a.it, nts, a.S, a.cbase);
  const bool any_src = s_pts[0] != 0, any_rec = s_pts[1] != 0;
  auto new_p = [&](int lx, int lz, T pold, T m0v, bool owned) -> T {
    const int gi2 = I0 - 1 + lx, gj2 = J0 - 1 + lz;
    if (gi2 < 0 || gi2 >= nx || gj2 < 0 || gj2 >= nz) return T(0);
    const int64_t c = (int64_t)gj2 * nx + gi2;
    T pv = pold;
    if (gi2 >= 1 && gi2 <= nx - 2 && gj2 >= 1 && gj2 <= nz - 2) {
      // update_p_CPML! (acoustic2D_VD_xPU.jl:17-37)
      T dvx = d4(s_vx[lz][lx], s_vx[lz][lx + 1], s_vx[lz][lx + 2], s_vx[lz][lx + 3]) * a.idx;
      if (gi2 <= h || gi2 >= nx - h - 1) {
        const int k = gi2 <= h ? gi2 : gi2 - nx + 2 * h + 2;
        const int64_t qx = (int64_t)s * a.sxx + (int64_t)gj2 * (2 * h + 2) + k;
        const T xi = cx.b(k) * a.xix_o[qx] + cx.a(k) * dvx;
        if (owned) a.xix_n[qx] = xi;
        dvx = dvx + xi;
      }
      T dvz = d4(s_vz[lz][lx], s_vz[lz + 1][lx], s_vz[lz + 2][lx], s_vz[lz + 3][lx]) * a.idz;
      if (gj2 <= h || gj2 >= nz - h - 1) {
        const int k = gj2 <= h ? gj2 : gj2 - nz + 2 * h + 2;
        const int64_t qz = (int64_t)s * a.sxz + (int64_t)k * nx + gi2;
        const T xi = cz.b(k) * a.xiz_o[qz] + cz.a(k) * dvz;
        if (owned) a.xiz_n[qz] = xi;
        dvz = dvz + xi;
      }
      pv = pv - m0v * (dvx + dvz);
    }
    // inject_sources! (acoustic2D_VD_xPU.jl:1-7), serial order per cell
    const int u = any_src ? find_point(a.pt.srow, a.pt.usrc_cell, a.pt.nrows, s, gj2, c) : -1;
    if (u >= 0) {
      const T *tf = a.srctf + a.pt.off_tf[s] + (a.it - 1);
      for (int k = a.pt.usrc_ptr[u]; k < a.pt.usrc_ptr[u + 1]; k++) pv += tf[(int64_t)nts * a.pt.usrc_list[k]];
    }
    if (owned) {
      st_nt(a.p_n + so + c, pv);
      if (sb >= 0) {
        st_nt(a.pbuf + (int64_t)(a.it - sb) * a.pslot + so + c, pv);
        if (a.smode == 1 && a.it == sb + 1) st_nt(a.pbuf + so + c, pold);
      }
      if (any_rec) {
        // record_receivers! (acoustic2D_VD_xPU.jl:9-15)
        const int r = find_point(a.pt.rrow, a.pt.urec_cell, a.pt.nrows, s, gj2, c);
        if (r >= 0) {
          T *tr = a.traces + a.pt.off_tr[s] + (a.it - 1);
          for (int k = a.pt.urec_ptr[r]; k < a.pt.urec_ptr[r + 1]; k++) tr[(int64_t)nts * a.pt.urec_list[k]] = pv;
        }
      }
    }
    return pv;
  };
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int lz = ty + BY * r + 1;
    s_p[lz][tx + 1] = new_p(tx + 1, lz, rp[r], rm0[r], true);
  }
#pragma unroll
  for (int k = 0; k < HR; k++)
    if (hlx[k] >= 0) s_p[hlz[k]][hlx[k]] = new_p(hlx[k], hlz[k], hp[k], hm0[k], false);
  __syncthreads();

  // ---- phase 2: update_vx_CPML! / update_vy_CPML! (:39-75) ---------------
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int lz = ty + BY * r;
    const int gj = J0 + lz;
    if (gi >= nx || gj >= nz) continue;
    const int64_t c = (int64_t)gj * nx + gi;
    if (gi <= nx - 2) {
      T d = d4(s_p[lz + 1][tx], s_p[lz + 1][tx + 1], s_p[lz + 1][tx + 2], s_p[lz + 1][tx + 3]) * a.idx;
      if (gi <= h - 1 || gi >= nx - h - 1) {
        const int k = gi <= h - 1 ? gi : gi + 1 - nx + 2 * h;
        const int64_t q = (int64_t)s * a.spx + (int64_t)gj * (2 * h) + k;
        const T ps = cx.bh(k) * a.psx_o[q] + cx.ah(k) * d;
        a.psx_n[q] = ps;
        d = d + ps;
      }
      st_nt(a.vx_n + so + c, s_vx[lz + 1][tx + 3] - rm1x[r] * d);
    }
    if (gj <= nz - 2) {
      T d = d4(s_p[lz][tx + 1], s_p[lz + 1][tx + 1], s_p[lz + 2][tx + 1], s_p[lz + 3][tx + 1]) * a.idz;
      if (gj <= h - 1 || gj >= nz - h - 1) {
        const int k = gj <= h - 1 ? gj : gj + 1 - nz + 2 * h;
        const int64_t q = (int64_t)s * a.spz + (int64_t)k * nx + gi;
        const T ps = cz.bh(k) * a.psz_o[q] + cz.ah(k) * d;
        a.psz_n[q] = ps;
        d = d + ps;
      }
      st_nt(a.vz_n + so + c, s_vz[lz + 3][tx + 1] - rm1z[r] * d);
    }
  }
}

// Forward / replay step: (p, vx, vz)^{it-1} -> (p, vx, vz)^{it}.  Interior
// tiles are stepped inline (FOLD, one launch per step) or left to
// vd2d_fwd_lean.
template <typename T, int TZ, bool FOLD>
__global__ __launch_bounds__(NT) void vd2d_fwd_kernel(Vd2dArgs<T> a) {
  int bx, bz, s;
  vd2d_tile_of(a, xcd_tile(blockIdx.x, gridDim.x), bx, bz, s);
  const int nts = a.nt_shot[s];
  if (a.it > nts || nts <= a.act_min) return;
  const int I0 = bx * TX, J0 = bz * TZ;
  __shared__ T s_vx[TZ + 3][TX + 6];   // vx^{it-1}: x in [I0-3, I0+TX+3), z in [J0-1, J0+TZ+2)
  __shared__ T s_vz[TZ + 6][TX + 3];   // vz^{it-1}: x in [I0-1, I0+TX+2), z in [J0-3, J0+TZ+3)
  __shared__ T s_p[TZ + 3][TX + 3];    // p^{it}:    x in [I0-1, I0+TX+2), z in [J0-1, J0+TZ+2)
  __shared__ int s_pts[2];
  if (vd2d_fwd_is_lean<TZ>(a, s, I0, J0)) {
    if (FOLD) {
      FwdTileModel<T, TZ> m;
      vd2d_fwd_lean_model<T, TZ>(a, I0, J0, m);
      vd2d_fwd_lean_tile<T, TZ>(a, s, nts, I0, J0, s_vx, s_vz, s_p, m);
    }
    return;
  }
  vd2d_fwd_general_tile<T, TZ>(a, s, nts, I0, J0, s_vx, s_vz, s_p, s_pts);
}

// Forward / replay step of a pair of shots (2k, 2k+1) per block: the model
// factors of an interior tile are read once for both shots (m0, m1x, m1z
// are 3 of the 9 values a cell step reads and writes).  The shots are
// stepped one after the other with the expressions of vd2d_fwd_kernel, so
// the results are bitwise the same.
template <typename T, int TZ>
__global__ __launch_bounds__(NT) void vd2d_fwd_pair_kernel(Vd2dArgs<T> a) {
  const int b = xcd_tile(blockIdx.x, gridDim.x);
  const int bx = b % a.nbx, bzs = b / a.nbx, bz = bzs % a.nbz, pr = bzs / a.nbz;
  const int I0 = bx * TX, J0 = bz * TZ;
  __shared__ T s_vx[TZ + 3][TX + 6];
  __shared__ T s_vz[TZ + 6][TX + 3];
  __shared__ T s_p[TZ + 3][TX + 3];
  __shared__ int s_pts[2];
  FwdTileModel<T, TZ> m;
  bool have_m = false;
  for (int k = 0; k < 2; k++) {
    const int s = 2 * pr + k;
    if (s >= a.nsh) break;
    const int nts = a.nt_shot[s];
    if (a.it > nts || nts <= a.act_min) continue;
    if (k == 1) __syncthreads();   // the LDS tiles of the first shot are consumed
    if (vd2d_fwd_is_lean<TZ>(a, s, I0, J0)) {
      if (!have_m) {
        vd2d_fwd_lean_model<T, TZ>(a, I0, J0, m);
        have_m = true;
      }
      vd2d_fwd_lean_tile<T, TZ>(a, s, nts, I0, J0, s_vx, s_vz, s_p, m);
    } else {
      vd2d_fwd_general_tile<T, TZ>(a, s, nts, I0, J0, s_vx, s_vz, s_p, s_pts);
    }
  }
}

// Two forward / replay steps in one launch: (p, vx, vz)^{it-1} ->
// (p, vx, vz)^{it+1}, with the intermediate level it kept on chip.
//
// A block owns a TX x TZ tile.  The velocities of step it+1 on the tile
// need the pressure p^{it+1} one cell left / two right (and up / down),
// which needs v^{it} three cells out, which needs p^{it} four cells out,
// which needs v^{it-1} six cells out.  So the block loads v^{it-1} and
// p^{it-1} on the enlarged rectangles, computes p^{it} on P1 = tile + 4
// (left/up) / 5 (right/down) in LDS, then v^{it} in place on its
// rectangles, then p^{it+1} in place on P2 = tile + 1 / 2, then v^{it+1}
// on the tile, which goes to HBM with p^{it+1} and the C-PML variables.
// Every cell update is the expression of vd2d_fwd_kernel (same operand
// order), so the results are bitwise those of two single steps.  C-PML
// memory variables are pointwise recurrences: a thread keeps the level-it
// value of each of its cells in a register and the same thread updates that
// cell again in the second step (P2 and the tile are walked in the P1 and
// v^{it} enumerations).  Per step the HBM traffic is about half that of a
// single-step launch; the redundant halo work is ~1.3x.
//
// A shot whose last step is it (nt_s == it) stores level it and stops after
// the first step.  The state is read from one buffer and written to the
// other, so the level written is it+1 (it for such a shot).
template <typename T, int TZ, int NB>
__global__ __launch_bounds__(NB) void vd2d_fwd2_kernel(Vd2dArgs<T> a) {
  constexpr int PX = TX + 9, PZ = TZ + 9;     // p:  x [I0-4, I0+TX+5), z [J0-4, J0+TZ+5)
  constexpr int AX = TX + 12, AZ = TZ + 9;    // vx: x [I0-6, I0+TX+6), z [J0-4, J0+TZ+5)
  constexpr int BX = TX + 9, BZ = TZ + 12;    // vz: x [I0-4, I0+TX+5), z [J0-6, J0+TZ+6)
  constexpr int X1X = TX + 6, X1Z = TZ + 3;   // vx^{it}: x [I0-3, I0+TX+3), z [J0-1, J0+TZ+2)
  constexpr int Z1X = TX + 3, Z1Z = TZ + 6;   // vz^{it}: x [I0-1, I0+TX+2), z [J0-3, J0+TZ+3)
  constexpr int NP = (PX * PZ + NB - 1) / NB;
  constexpr int NVX = (X1X * X1Z + NB - 1) / NB, NVZ = (Z1X * Z1Z + NB - 1) / NB;
  const int b = xcd_tile(blockIdx.x, gridDim.x);
  const int bx = b % a.nbx, bzs = b / a.nbx, bz = bzs % a.nbz, s = bzs / a.nbz;
  const int nts = a.nt_shot[s];
  if (a.it > nts || nts <= a.act_min) return;
  const bool two = a.it + 1 <= nts;
  const int nx = a.nx, nz = a.nz, h = a.h;
  const int I0 = bx * TX, J0 = bz * TZ;
  const int tid = threadIdx.y * TX + threadIdx.x;
  const int64_t so = (int64_t)s * a.N;
  const T *cb = a.cpml + (int64_t)s * a.cstride;
  const AxisCoef<T> cx = axis_coef(cb, h, 0), cz = axis_coef(cb, h, 1);

  __shared__ T s_vx[AZ][AX];
  __shared__ T s_vz[BZ][BX];
  __shared__ T s_p[PZ][PX];
  __shared__ int s_pts[2];
  if (tid == 0) {
    const int *sr = a.pt.srow + (int64_t)s * (a.pt.nrows + 1);
    const int *rr = a.pt.rrow + (int64_t)s * (a.pt.nrows + 1);
    s_pts[0] = sr[max(J0 - 4, 0)] < sr[min(J0 + TZ + 5, nz)];
    s_pts[1] = a.traces != nullptr && rr[min(J0, nz)] < rr[min(J0 + TZ, nz)];
  }

  // ---- loads: v^{it-1}, p^{it-1} into LDS; factors and C-PML variables of
  // this thread's cells into registers ------------------------------------
  // all global loads of a thread are issued before its first LDS store
  constexpr int KA = (AZ * AX + NB - 1) / NB, KB = (BZ * BX + NB - 1) / NB;
  T ga[KA], gb[KB];
#pragma unroll
  for (int k = 0; k < KA; k++) {
    const int q = tid + k * NB;
    const int lz = q / AX, lx = q % AX;
    const int gi = I0 - 6 + lx, gj = J0 - 4 + lz;
    T v = 0;
    if (q < AZ * AX && gi >= 0 && gi <= nx - 2 && gj >= 0 && gj <= nz - 1) v = a.vx_o[so + (int64_t)gj * nx + gi];
    ga[k] = v;
  }
#pragma unroll
  for (int k = 0; k < KB; k++) {
    const int q = tid + k * NB;
    const int lz = q / BX, lx = q % BX;
    const int gi = I0 - 4 + lx, gj = J0 - 6 + lz;
    T v = 0;
    if (q < BZ * BX && gi >= 0 && gi <= nx - 1 && gj >= 0 && gj <= nz - 2) v = a.vz_o[so + (int64_t)gj * nx + gi];
    gb[k] = v;
  }
  T rm0[NP], rxx[NP], rxz[NP];
#pragma unroll
  for (int k = 0; k < NP; k++) {
    const int q = tid + k * NB;
    const int pz = q / PX, px = q % PX;
    const int gi = I0 - 4 + px, gj = J0 - 4 + pz;
    T vp = 0, vm = 0, x0 = 0, x1 = 0;
    if (q < PX * PZ && gi >= 0 && gi <= nx - 1 && gj >= 0 && gj <= nz - 1) {
      const int64_t c = (int64_t)gj * nx + gi;
      vp = a.p_o[so + c];
      vm = a.m0[c];
      if (gi >= 1 && gi <= nx - 2 && gj >= 1 && gj <= nz - 2) {
        if (gi <= h || gi >= nx - h - 1) {
          const int kk = gi <= h ? gi : gi - nx + 2 * h + 2;
          x0 = a.xix_o[(int64_t)s * a.sxx + (int64_t)gj * (2 * h + 2) + kk];
        }
        if (gj <= h || gj >= nz - h - 1) {
          const int kk = gj <= h ? gj : gj - nz + 2 * h + 2;
          x1 = a.xiz_o[(int64_t)s * a.sxz + (int64_t)kk * nx + gi];
        }
      }
    }
    if (q < PX * PZ) s_p[pz][px] = vp;
    rm0[k] = vm;
    rxx[k] = x0;
    rxz[k] = x1;
  }
  T rm1x[NVX], rpx[NVX];
#pragma unroll
  for (int k = 0; k < NVX; k++) {
    const int q = tid + k * NB;
    const int gi = I0 - 3 + q % X1X, gj = J0 - 1 + q / X1X;
    T vm = 0, ps = 0;
    if (q < X1X * X1Z && gi >= 0 && gi <= nx - 2 && gj >= 0 && gj <= nz - 1) {
      vm = a.m1x[(int64_t)gj * nx + gi];
      if (gi <= h - 1 || gi >= nx - h - 1) {
        const int kk = gi <= h - 1 ? gi : gi + 1 - nx + 2 * h;
        ps = a.psx_o[(int64_t)s * a.spx + (int64_t)gj * (2 * h) + kk];
      }
    }
    rm1x[k] = vm;
    rpx[k] = ps;
  }
  T rm1z[NVZ], rpz[NVZ];
#pragma unroll
  for (int k = 0; k < NVZ; k++) {
    const int q = tid + k * NB;
    const int gi = I0 - 1 + q % Z1X, gj = J0 - 3 + q / Z1X;
    T vm = 0, ps = 0;
    if (q < Z1X * Z1Z && gi >= 0 && gi <= nx - 1 && gj >= 0 && gj <= nz - 2) {
      vm = a.m1z[(int64_t)gj * nx + gi];
      if (gj <= h - 1 || gj >= nz - h - 1) {
        const int kk = gj <= h - 1 ? gj : gj + 1 - nz + 2 * h;
        ps = a.psz_o[(int64_t)s * a.spz + (int64_t)kk * nx + gi];
      }
    }
    rm1z[k] = vm;
    rpz[k] = ps;
  }
#pragma unroll
  for (int k = 0; k < KA; k++) {
    const int q = tid + k * NB;
    if (q < AZ * AX) s_vx[q / AX][q % AX] = ga[k];
  }
#pragma unroll
  for (int k = 0; k < KB; k++) {
    const int q = tid + k * NB;
    if (q < BZ * BX) s_vz[q / BX][q % BX] = gb[k];
  }
  __syncthreads();

  const bool any_src = s_pts[0] != 0, any_rec = s_pts[1] != 0;
  // pressure update of step `st` at this thread's P1 cells (inner: P2 only),
  // in place in s_p (update_p_CPML! + inject_sources!, then the tile's
  // recording, history and, when `fin`, the final state)
  auto p_phase = [&](int st, bool inner, bool fin) {
    const int sb = store_base(a.smode, st, nts, a.S, a.cbase);
#pragma unroll
    for (int k = 0; k < NP; k++) {
      const int q = tid + k * NB;
      const int pz = q / PX, px = q % PX;
      if (q >= PX * PZ) continue;
      if (inner && (px < 3 || px >= TX + 6 || pz < 3 || pz >= TZ + 6)) continue;
      const int gi = I0 - 4 + px, gj = J0 - 4 + pz;
      if (gi < 0 || gi >= nx || gj < 0 || gj >= nz) continue;   // stays 0
      const int64_t c = (int64_t)gj * nx + gi;
      const T pold = s_p[pz][px];
      T pv = pold;
      if (gi >= 1 && gi <= nx - 2 && gj >= 1 && gj <= nz - 2) {
        T dvx = d4(s_vx[pz][px], s_vx[pz][px + 1], s_vx[pz][px + 2], s_vx[pz][px + 3]) * a.idx;
        if (gi <= h || gi >= nx - h - 1) {
          const int kk = gi <= h ? gi : gi - nx + 2 * h + 2;
          const T xi = cx.b(kk) * rxx[k] + cx.a(kk) * dvx;
          rxx[k] = xi;
          dvx = dvx + xi;
        }
        T dvz = d4(s_vz[pz][px], s_vz[pz + 1][px], s_vz[pz + 2][px], s_vz[pz + 3][px]) * a.idz;
        if (gj <= h || gj >= nz - h - 1) {
          const int kk = gj <= h ? gj : gj - nz + 2 * h + 2;
          const T xi = cz.b(kk) * rxz[k] + cz.a(kk) * dvz;
          rxz[k] = xi;
          dvz = dvz + xi;
        }
        pv = pv - rm0[k] * (dvx + dvz);
      }
      const int u = any_src ? find_point(a.pt.srow, a.pt.usrc_cell, a.pt.nrows, s, gj, c) : -1;
      if (u >= 0) {
        const T *tf = a.srctf + a.pt.off_tf[s] + (st - 1);
        for (int e = a.pt.usrc_ptr[u]; e < a.pt.usrc_ptr[u + 1]; e++) pv += tf[(int64_t)nts * a.pt.usrc_list[e]];
      }
      s_p[pz][px] = pv;
      const bool owned = px >= 4 && px < TX + 4 && pz >= 4 && pz < TZ + 4;
      if (owned) {
        if (sb >= 0) {
          a.pbuf[(int64_t)(st - sb) * a.pslot + so + c] = pv;
          if (a.smode == 1 && st == sb + 1) a.pbuf[so + c] = pold;
        }
        if (any_rec) {
          const int r = find_point(a.pt.rrow, a.pt.urec_cell, a.pt.nrows, s, gj, c);
          if (r >= 0) {
            T *tr = a.traces + a.pt.off_tr[s] + (st - 1);
            for (int e = a.pt.urec_ptr[r]; e < a.pt.urec_ptr[r + 1]; e++) tr[(int64_t)nts * a.pt.urec_list[e]] = pv;
          }
        }
        if (fin) {
          a.p_n[so + c] = pv;
          if (gi >= 1 && gi <= nx - 2 && gj >= 1 && gj <= nz - 2) {
            if (gi <= h || gi >= nx - h - 1) {
              const int kk = gi <= h ? gi : gi - nx + 2 * h + 2;
              a.xix_n[(int64_t)s * a.sxx + (int64_t)gj * (2 * h + 2) + kk] = rxx[k];
            }
            if (gj <= h || gj >= nz - h - 1) {
              const int kk = gj <= h ? gj : gj - nz + 2 * h + 2;
              a.xiz_n[(int64_t)s * a.sxz + (int64_t)kk * nx + gi] = rxz[k];
            }
          }
        }
      }
    }
  };
  // velocity update at this thread's v^{it} cells (inner: the tile only),
  // in place in s_vx / s_vz, or to HBM when `fin`
  auto v_phase = [&](bool inner, bool fin) {
#pragma unroll
    for (int k = 0; k < NVX; k++) {
      const int q = tid + k * NB;
      const int az = q / X1X, ax = q % X1X;
      if (q >= X1X * X1Z) continue;
      if (inner && (ax < 3 || ax >= TX + 3 || az < 1 || az >= TZ + 1)) continue;
      const int gi = I0 - 3 + ax, gj = J0 - 1 + az;
      if (gi < 0 || gi > nx - 2 || gj < 0 || gj > nz - 1) continue;   // stays 0
      T d = d4(s_p[az + 3][ax], s_p[az + 3][ax + 1], s_p[az + 3][ax + 2], s_p[az + 3][ax + 3]) * a.idx;
      const bool strip = gi <= h - 1 || gi >= nx - h - 1;
      const int kk = gi <= h - 1 ? gi : gi + 1 - nx + 2 * h;
      if (strip) {
        const T ps = cx.bh(kk) * rpx[k] + cx.ah(kk) * d;
        rpx[k] = ps;
        d = d + ps;
      }
      const T v = s_vx[az + 3][ax + 3] - rm1x[k] * d;
      const bool owned = ax >= 3 && ax < TX + 3 && az >= 1 && az < TZ + 1;
      if (fin) {
        if (owned) {
          const int64_t c = (int64_t)gj * nx + gi;
          a.vx_n[so + c] = v;
          if (strip) a.psx_n[(int64_t)s * a.spx + (int64_t)gj * (2 * h) + kk] = rpx[k];
        }
      } else {
        s_vx[az + 3][ax + 3] = v;
      }
    }
#pragma unroll
    for (int k = 0; k < NVZ; k++) {
      const int q = tid + k * NB;
      const int bz2 = q / Z1X, bx2 = q % Z1X;
      if (q >= Z1X * Z1Z) continue;
      if (inner && (bx2 < 1 || bx2 >= TX + 1 || bz2 < 3 || bz2 >= TZ + 3)) continue;
      const int gi = I0 - 1 + bx2, gj = J0 - 3 + bz2;
      if (gi < 0 || gi > nx - 1 || gj < 0 || gj > nz - 2) continue;   // stays 0
      T d = d4(s_p[bz2][bx2 + 3], s_p[bz2 + 1][bx2 + 3], s_p[bz2 + 2][bx2 + 3], s_p[bz2 + 3][bx2 + 3]) * a.idz;
      const bool strip = gj <= h - 1 || gj >= nz - h - 1;
      const int kk = gj <= h - 1 ? gj : gj + 1 - nz + 2 * h;
      if (strip) {
        const T ps = cz.bh(kk) * rpz[k] + cz.ah(kk) * d;
        rpz[k] = ps;
        d = d + ps;
      }
      const T v = s_vz[bz2 + 3][bx2 + 3] - rm1z[k] * d;
      const bool owned = bx2 >= 1 && bx2 < TX + 1 && bz2 >= 3 && bz2 < TZ + 3;
      if (fin) {
        if (owned) {
          const int64_t c = (int64_t)gj * nx + gi;
          a.vz_n[so + c] = v;
          if (strip) a.psz_n[(int64_t)s * a.spz + (int64_t)kk * nx + gi] = rpz[k];
        }
      } else {
        s_vz[bz2 + 3][bx2 + 3] = v;
      }
    }
  };

  p_phase(a.it, false, !two);   // p^{it} on P1
  __syncthreads();
  if (!two) {
    v_phase(true, true);        // v^{it} on the tile, to HBM
    return;
  }
  v_phase(false, false);        // v^{it} on its rectangles, in LDS
  __syncthreads();
  p_phase(a.it + 1, true, true);   // p^{it+1} on P2
  __syncthreads();
  v_phase(true, true);          // v^{it+1} on the tile, to HBM
}

// ---------------------------------------------------------------------------
// Several levels per launch (vd2d_stepn_kernel).
//
// A block of NW waves holds a 64 x (NW R) window of pressure, velocities and
// model factors in registers (lane = column, R rows per wave) and steps it n
// times.  A level reaches three cells to every side (pressure from velocities
// two cells before and one after, velocities from the new pressure one before
// and two after), so the block owns, and writes, the cells at least 3 n from
// the window's sides (all cells up to a side that is the grid's).  x
// neighbours come from the adjacent lanes, z neighbours from the thread's own
// rows; the last two and the first velocity row of each wave, then the last
// and the first two pressure rows, pass through LDS: two barriers per level.
// The C-PML memory variables of the strip cells step along in registers; point
// values of the n levels are staged in LDS once.  Cell updates are spelled as
// in vd2d_fwd_general_tile: results are bitwise those of n single steps.
//
// Bound by latency on small grids (701 x 403 float32: 18 us for 5 levels, 9.7 us
// for one of the tile steps; 1.5 waves per SIMD) and by what the windows step
// twice on large ones, 2.1 times the owned cells (96 rows, 4 levels): 1000 x
// 700, 8 shots float32 49 -> 32 us per level; 2000 x 800, 32 shots 349 -> 254.
// Counters there (64 shots), forward / adjoint: vector units issue 0.56 / 0.36
// of the time at 3.5 / 1.8 waves per SIMD, 2.7 / 3.3 TB/s, 1.31 / 1.47 times the
// bytes of the owned cells.
// The adjoint keeps the three gradients of its cells in registers too and
// reads one history level per level: 701 x 403 10.9 -> 5.1 us, 2000 x 800, 32
// shots 585 -> 474 (8 x 8 rows; 4 x 16, where six registers spill, takes 1.13
// times as long).
template <typename T, int R, int NW>
struct Vd2dNLds : LevelPoints<T, NW * R> {
  T vz[3][NW][TX];             // rows R-2, R-1 and 0 of vz
  T p[3][NW][TX];              // rows R-1, 0 and 1 of the new pressure
  T cz[NW * R][4];             // z C-PML coefficients b, a (pressure), b_h, a_h (velocity) of the rows
};

// Registers of one thread: R cells of a column.
template <typename T, int R>
struct Vd2dNRegs {
  T p[R], vx[R], vz[R], m0[R], m1x[R], m1z[R];
  T xix[R], xiz[R], psx[R], psz[R];
};

// Pressure of one level; vu2, vu1: vz of the two rows before the wave's, vd of
// the one after.  XS: the window reaches an x strip or side; ZS: the wave's
// rows reach a z strip or side.
template <typename T, int R, int NW, bool XS, bool ZS>
__device__ __forceinline__ void vd2d_n_pressure(const Vd2dArgs<T> &a, const Vd2dNLds<T, R, NW> &L, const LevelWin &W,
                                                bool xst, const T *xc, T vu2, T vu1, T vd, Vd2dNRegs<T, R> &G) {
  const bool xin = !XS || (W.i >= 1 && W.i <= a.nx - 2);
#pragma unroll
  for (int r = 0; r < R; r++) {
    const T x0 = G.vx[r], x1 = lane_before(x0), x2 = lane_before(x1);
    T dvx = d4(x2, x1, x0, lane_after(x0)) * a.idx;
    T dvz = d4(r > 1 ? G.vz[r > 1 ? r - 2 : 0] : r > 0 ? vu1 : vu2, r > 0 ? G.vz[r > 0 ? r - 1 : 0] : vu1, G.vz[r],
               r + 1 < R ? G.vz[r + 1 < R ? r + 1 : r] : vd) * a.idz;
    const bool interior = xin && (!ZS || (W.jin >> r & 1));
    if (XS) {
      const T xi = xc[0] * G.xix[r] + xc[1] * dvx;
      if (xst && interior) {
        G.xix[r] = xi;
        dvx = dvx + xi;
      }
    }
    if (ZS) {
      if (W.xzr >> r & 1) {
        const T *c = L.cz[W.w * R + r];
        const T xi = c[0] * G.xiz[r] + c[1] * dvz;
        if (interior) {
          G.xiz[r] = xi;
          dvz = dvz + xi;
        }
      }
    }
    const T pv = G.p[r] - G.m0[r] * (dvx + dvz);
    G.p[r] = interior ? pv : G.p[r];
  }
}

// Velocities of one level; pu: new pressure of the row before the wave's, pd1,
// pd2 of the two after.
template <typename T, int R, int NW, bool XS, bool ZS>
__device__ __forceinline__ void vd2d_n_velocity(const Vd2dArgs<T> &a, const Vd2dNLds<T, R, NW> &L, const LevelWin &W,
                                                bool pst, const T *xc, T pu, T pd1, T pd2, Vd2dNRegs<T, R> &G) {
  const bool xv = !XS || W.i <= a.nx - 2, xg = !XS || W.i <= a.nx - 1;
#pragma unroll
  for (int r = 0; r < R; r++) {
    const T p0 = G.p[r], p1 = lane_after(p0), p2 = lane_after(p1);
    T dx = d4(lane_before(p0), p0, p1, p2) * a.idx;
    T dz = d4(r > 0 ? G.p[r > 0 ? r - 1 : 0] : pu, p0, r + 1 < R ? G.p[r + 1 < R ? r + 1 : r] : pd1,
              r + 2 < R ? G.p[r + 2 < R ? r + 2 : r] : r + 1 < R ? pd1 : pd2) * a.idz;
    if (XS) {
      const T ps = xc[2] * G.psx[r] + xc[3] * dx;
      if (pst) {
        G.psx[r] = ps;
        dx = dx + ps;
      }
    }
    if (ZS) {
      if (W.kzr >> r & 1) {
        const T *c = L.cz[W.w * R + r];
        const T ps = c[2] * G.psz[r] + c[3] * dz;
        G.psz[r] = ps;
        dz = dz + ps;
      }
    }
    const T vx = G.vx[r] - G.m1x[r] * dx, vz = G.vz[r] - G.m1z[r] * dz;
    G.vx[r] = xv && (!ZS || (W.jg >> r & 1)) ? vx : G.vx[r];
    G.vz[r] = xg && (!ZS || (W.jv >> r & 1)) ? vz : G.vz[r];
  }
}

// Correlation of one adjoint level (correlate_gradient_xPU.jl:12-21,
// acoustic2D_VD_xPU.jl:180-198): cur, prev: the replayed pressure of the level
// and the one before, rows from the one before the thread's to two after.
// EDGE: the window or the rows reach a side of the grid.
template <typename T, int R, bool EDGE>
__device__ __forceinline__ void vd2d_n_correlate(const Vd2dArgs<T> &a, const LevelWin &W, const T *cur, const T *prev,
                                                 const Vd2dNRegs<T, R> &G, T *g0, T *g1x, T *g1z) {
  T c[R + 3];
#pragma unroll
  for (int q = 0; q < R + 3; q++) {
    const int j = W.j0 - 1 + q;
    c[q] = EDGE && (W.i > a.nx - 1 || j < 0 || j > a.nz - 1) ? T(0) : cur[q];
  }
#pragma unroll
  for (int r = 0; r < R; r++) {
    const T pcv = c[r + 1];
    g0[r] = g0[r] - (G.p[r] * (pcv - prev[r + 1]) * a.idt);
    const T p1 = lane_after(pcv);
    const T dpx = d4(lane_before(pcv), pcv, p1, lane_after(p1)) * a.idx;
    g1x[r] = g1x[r] + G.vx[r] * dpx;
    const T dpz = d4(c[r], pcv, c[r + 2], c[r + 3]) * a.idz;
    g1z[r] = g1z[r] + G.vz[r] * dpz;
  }
}

// Forward / replay levels it .. it+n-1, or (ADJ) adjoint levels it .. it-n+1:
// velocities from the old pressure, then the pressure, residual injection and
// the correlation with the replayed pressure, which is loaded a level ahead.
template <typename T, int R, int NW, bool ADJ>
__global__ __launch_bounds__(NW *TX, NW / 4) void vd2d_stepn_kernel(Vd2dArgs<T> a, int n) {
  __shared__ Vd2dNLds<T, R, NW> L;
  constexpr int H = NW * R;
  if (threadIdx.x == 0) L.used = L.rused = 0;
  __syncthreads();
  const int b = xcd_tile(blockIdx.x, gridDim.x);
  const int t = b / a.nbx;
  const int bx = b - t * a.nbx, by = t % a.nbz, s = t / a.nbz;
  const int nts = a.nt_shot[s];
  const int nx = a.nx, nz = a.nz, h = a.h;
  const int X0 = bx * (TX - 6 * n), Z0 = by * (H - 6 * n);
  LevelWin W;
  W.lane = threadIdx.x & (TX - 1);
  W.w = __builtin_amdgcn_readfirstlane(threadIdx.x / TX);
  W.i = X0 + W.lane;
  W.j0 = Z0 + W.w * R;
  W.own = W.i < nx && W.lane >= (bx ? 3 * n : 0) && W.lane < (bx < a.nbx - 1 ? TX - 3 * n : TX);
  W.rows = W.jin = W.kzr = W.xzr = W.jg = W.jv = 0;
  const int own0 = by ? Z0 + 3 * n : 0, own1 = by < a.nbz - 1 ? Z0 + H - 3 * n : nz;
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int j = W.j0 + r;
    if (j >= own0 && j < own1) W.rows |= 1 << r;
    if (j < nz) W.jg |= 1 << r;
    if (j <= nz - 2) W.jv |= 1 << r;
    if (j >= 1 && j <= nz - 2) {
      W.jin |= 1 << r;
      if (j <= h || j >= nz - h - 1) W.xzr |= 1 << r;
    }
    if (j < h || (j >= nz - h - 1 && j <= nz - 2)) W.kzr |= 1 << r;
  }
  const int64_t so = (int64_t)s * a.N;
  const bool xs = X0 <= max(h, 1) || X0 + TX - 1 >= nx - h - 1;
  // (without strips too, two rows before the last one: the correlation reads
  // the pressure two rows on, zero beyond the grid)
  const bool zs = W.j0 <= max(h, 1) || W.j0 + R - 1 >= nz - max(h, 1) - 1;
  // strip entries of the column: pressure (xi), velocity (psi)
  const bool xst = W.i >= 1 && W.i <= nx - 2 && (W.i <= h || W.i >= nx - h - 1);
  const bool pst = W.i < h || (W.i >= nx - h - 1 && W.i <= nx - 2);
  const int kxi = xst ? (W.i <= h ? W.i : W.i - nx + 2 * h + 2) : 0, kps = pst ? (W.i < h ? W.i : W.i + 1 - nx + 2 * h) : 0;

  // Fields and factors, zero outside their grids (the derivative rule).
  Vd2dNRegs<T, R> G;
  const unsigned ic = min(W.i, nx - 1);
  auto row = [&](const T *p, int r) { return p + (int64_t)min(W.j0 + r, nz - 1) * nx; };
#pragma unroll
  for (int r = 0; r < R; r++) {
    G.p[r] = row(a.p_o + so, r)[ic];
    G.vx[r] = row(a.vx_o + so, r)[ic];
    G.vz[r] = row(a.vz_o + so, r)[ic];
    G.m0[r] = row(a.m0, r)[ic];
    G.m1x[r] = row(a.m1x, r)[ic];
    G.m1z[r] = row(a.m1z, r)[ic];
    G.xix[r] = G.xiz[r] = G.psx[r] = G.psz[r] = T(0);
  }
  auto zxi = [&](int r) { return W.j0 + r <= h ? W.j0 + r : W.j0 + r - nz + 2 * h + 2; };
  auto zps = [&](int r) { return W.j0 + r < h ? W.j0 + r : W.j0 + r + 1 - nz + 2 * h; };
  T xc[4] = {T(0), T(0), T(0), T(0)};
  if (xs && h > 0) {
    const AxisCoef<T> cx = axis_coef(a.cpml + (int64_t)s * a.cstride, h, 0);
    const T c0 = cx.b(kxi), c1 = cx.a(kxi), c2 = cx.bh(kps), c3 = cx.ah(kps);
    xc[0] = c0;
    xc[1] = c1;
    xc[2] = c2;
    xc[3] = c3;
#pragma unroll
    for (int r = 0; r < R; r++) {
      const int64_t j = min(W.j0 + r, nz - 1);
      G.xix[r] = (a.xix_o + (int64_t)s * a.sxx + j * (2 * h + 2))[(unsigned)kxi];
      G.psx[r] = (a.psx_o + (int64_t)s * a.spx + j * (2 * h))[(unsigned)kps];
    }
  }
  if (zs) {
#pragma unroll
    for (int r = 0; r < R; r++) {
      if (W.xzr >> r & 1) G.xiz[r] = (a.xiz_o + (int64_t)s * a.sxz + (int64_t)zxi(r) * nx)[ic];
      if (W.kzr >> r & 1) G.psz[r] = (a.psz_o + (int64_t)s * a.spz + (int64_t)zps(r) * nx)[ic];
    }
  }
  T g0[ADJ ? R : 1], g1x[ADJ ? R : 1], g1z[ADJ ? R : 1];
  if constexpr (ADJ) {
#pragma unroll
    for (int r = 0; r < R; r++) {
      g0[r] = row(a.g0 + so, r)[ic];
      g1x[r] = row(a.g1x + so, r)[ic];
      g1z[r] = row(a.g1z + so, r)[ic];
    }
  }
  // Levels of this shot: a forward one ends at nts, an adjoint one starts there
  // (from zero fields).  Tested after the loads above were issued, so that
  // they do not wait for nts.
  const int la = ADJ ? min(a.it, nts) : a.it;
  const int nl = ADJ ? la - (a.it - n) : min(n, nts - a.it + 1);
  if (nl <= 0 || nts <= a.act_min) return;
  T d0[ADJ ? R + 3 : 1], d1[ADJ ? R + 3 : 1];      // replayed pressure of a level, rows j0-1 .. j0+R+1
  auto fetch = [&](T *d, int l) {
    const T *slot = a.pbuf + (int64_t)(max(l, a.cbase) - a.cbase) * a.pslot + so;
#pragma unroll
    for (int q = 0; q < R + 3; q++) d[q] = (slot + (int64_t)min(max(W.j0 - 1 + q, 0), nz - 1) * nx)[ic];
  };
  if constexpr (ADJ) {
    fetch(d0, la);
    fetch(d1, la - 1);
  }
  if (xs || zs) {
#pragma unroll
    for (int r = 0; r < R; r++) {
      const bool g = W.i < nx && (W.jg >> r & 1);
      G.p[r] = g ? G.p[r] : T(0);
      G.vx[r] = g && W.i <= nx - 2 ? G.vx[r] : T(0);
      G.vz[r] = g && (W.jv >> r & 1) ? G.vz[r] : T(0);
    }
  }
  const int64_t otr = a.pt.off_tr[s];     // (here: a load in the level loop would wait for the wave's stores)
  level_points<T, R, ADJ>(a, L, W, s, nts, X0, la, nl);
  if (threadIdx.x < H) {
    const int j = Z0 + (int)threadIdx.x;
    const AxisCoef<T> cz = axis_coef(a.cpml + (int64_t)s * a.cstride, h, 1);
    T *q = L.cz[threadIdx.x];
    const bool x = j >= 1 && j <= nz - 2 && (j <= h || j >= nz - h - 1), v = j < h || (j >= nz - h - 1 && j <= nz - 2);
    const int kx = j <= h ? j : j - nz + 2 * h + 2, kv = j < h ? j : j + 1 - nz + 2 * h;
    q[0] = x ? cz.b(kx) : T(0);
    q[1] = x ? cz.a(kx) : T(0);
    q[2] = v ? cz.bh(kv) : T(0);
    q[3] = v ? cz.ah(kv) : T(0);
  }
  // level l > seg0 >= 0 goes to slot l - seg0
  const int seg0 = ADJ ? -1 : store_base(a.smode, 1 << 30, nts, a.S, a.cbase);

  auto pressure = [&] {
    const int wu = W.w > 0 ? W.w - 1 : 0, wd = W.w < NW - 1 ? W.w + 1 : NW - 1;
    L.vz[0][W.w][W.lane] = G.vz[R - 2];
    L.vz[1][W.w][W.lane] = G.vz[R - 1];
    L.vz[2][W.w][W.lane] = G.vz[0];
    __syncthreads();
    // (beyond the window: zero, what the grid's own sides need)
    T vu2 = L.vz[0][wu][W.lane], vu1 = L.vz[1][wu][W.lane], vd = L.vz[2][wd][W.lane];
    if (W.w == 0) vu2 = vu1 = T(0);
    if (W.w == NW - 1) vd = T(0);
    if (xs) vd2d_n_pressure<T, R, NW, true, true>(a, L, W, xst, xc, vu2, vu1, vd, G);
    else if (zs) vd2d_n_pressure<T, R, NW, false, true>(a, L, W, xst, xc, vu2, vu1, vd, G);
    else vd2d_n_pressure<T, R, NW, false, false>(a, L, W, xst, xc, vu2, vu1, vd, G);
  };
  auto velocity = [&] {
    const int wu = W.w > 0 ? W.w - 1 : 0, wd = W.w < NW - 1 ? W.w + 1 : NW - 1;
    L.p[0][W.w][W.lane] = G.p[R - 1];
    L.p[1][W.w][W.lane] = G.p[0];
    L.p[2][W.w][W.lane] = G.p[1];
    __syncthreads();
    T pu = L.p[0][wu][W.lane], pd1 = L.p[1][wd][W.lane], pd2 = L.p[2][wd][W.lane];
    if (W.w == 0) pu = T(0);
    if (W.w == NW - 1) pd1 = pd2 = T(0);
    if (xs) vd2d_n_velocity<T, R, NW, true, true>(a, L, W, pst, xc, pu, pd1, pd2, G);
    else if (zs) vd2d_n_velocity<T, R, NW, false, true>(a, L, W, pst, xc, pu, pd1, pd2, G);
    else vd2d_n_velocity<T, R, NW, false, false>(a, L, W, pst, xc, pu, pd1, pd2, G);
  };
  // injection and (forward) recording of level l, number m
  auto points = [&](int m, int l) {
    if (!(W.imask | W.rmask)) return;
#pragma unroll
    for (int r = 0; r < R; r++) {
      if (W.imask >> r & 1) {
        T inj = 0;
        level_inject<T, R, ADJ>(a, L, W, s, nts, r, m, l, G.m0[r], G.p[r], inj);
      }
      if (!ADJ && (W.rmask & W.rows) >> r & 1 && W.own)
        level_record<T, R>(a, L, W, nts, r, a.traces + otr + (l - 1), G.p[r]);
    }
  };
  auto fresh = [&] {
    opaque(W.j0);
    opaque(W.rows);
    opaque(W.jin);
    opaque(W.kzr);
    opaque(W.xzr);
    opaque(W.jg);
    opaque(W.jv);
    opaque(W.imask);
    opaque(W.rmask);
  };
  if constexpr (ADJ) {
    auto level = [&](int m, T *cur, const T *prev) {
      fresh();
      velocity();
      pressure();
      points(m, la - m);
      if (xs || zs) vd2d_n_correlate<T, R, true>(a, W, cur, prev, G, g0, g1x, g1z);
      else vd2d_n_correlate<T, R, false>(a, W, cur, prev, G, g0, g1x, g1z);
      fetch(cur, la - m - 2);
    };
#pragma clang loop unroll(disable)
    for (int m = 0; m < nl; m += 2) {
      level(m, d0, d1);
      if (m + 1 < nl) level(m + 1, d1, d0);
    }
  } else {
#pragma clang loop unroll(disable)
    for (int m = 0; m < nl; m++) {
      fresh();
      const int l = a.it + m;
      if (seg0 >= 0 && a.smode == 1 && l == seg0 + 1 && W.own) {
#pragma unroll
        for (int r = 0; r < R; r++)
          if (W.rows >> r & 1) (a.pbuf + so + (int64_t)(W.j0 + r) * nx)[ic] = G.p[r];
      }
      pressure();
      points(m, l);
      velocity();
      if (seg0 >= 0 && l > seg0 && W.own) {
        T *hs = a.pbuf + (int64_t)(l - seg0) * a.pslot + so;
#pragma unroll
        for (int r = 0; r < R; r++)
          if (W.rows >> r & 1) st_nt(hs + (int64_t)(W.j0 + r) * nx + ic, G.p[r]);
      }
    }
  }

  if (!W.own) return;
#pragma unroll
  for (int r = 0; r < R; r++) {
    if (!(W.rows >> r & 1)) continue;
    const int64_t j = W.j0 + r, o = so + j * nx;
    (a.p_n + o)[ic] = G.p[r];
    if (W.i <= nx - 2) (a.vx_n + o)[ic] = G.vx[r];
    if (j <= nz - 2) (a.vz_n + o)[ic] = G.vz[r];
    if (xst) (a.xix_n + (int64_t)s * a.sxx + j * (2 * h + 2))[(unsigned)kxi] = G.xix[r];
    if (pst) (a.psx_n + (int64_t)s * a.spx + j * (2 * h))[(unsigned)kps] = G.psx[r];
    if (W.xzr >> r & 1) (a.xiz_n + (int64_t)s * a.sxz + (int64_t)zxi(r) * nx)[ic] = G.xiz[r];
    if (W.kzr >> r & 1) (a.psz_n + (int64_t)s * a.spz + (int64_t)zps(r) * nx)[ic] = G.psz[r];
    if constexpr (ADJ) {
      (a.g0 + o)[ic] = g0[r];
      if (W.i <= nx - 2) (a.g1x + o)[ic] = g1x[r];
      if (j <= nz - 2) (a.g1z + o)[ic] = g1z[r];
    }
  }
}

// Forward / replay step marching down z.  A block owns a strip of 64*W
// columns and a chunk of rows [Z0, Z1) and walks it row by row: the new
// pressure of row j (and of the one-left / two-right halo columns the
// velocity update needs) is computed from LDS rings of old vx and vz rows,
// then the velocities of row j-2, whose pressure rows j-3..j are now in the
// ring of new pressures.  Every input row is read once per block (only the
// three rows above and below a chunk are read twice), and the loads of row
// j+1 are issued before the work on row j.  Ring depths are one row more
// than a step reads, so two barriers per row suffice.
template <typename T, int W>
__global__ __launch_bounds__(64 * W) void vd2d_fwd_march(Vd2dArgs<T> a) {
  constexpr int TXM = 64 * W;
  const int b = xcd_tile(blockIdx.x, gridDim.x);
  const int bx = b % a.nbx, bzs = b / a.nbx, bz = bzs % a.nbz, s = bzs / a.nbz;
  const int nts = a.nt_shot[s];
  if (a.it > nts || nts <= a.act_min) return;
  const int nx = a.nx, nz = a.nz, h = a.h;
  const int I0 = bx * TXM, Z0 = bz * a.ch, Z1 = min(Z0 + a.ch, nz);
  const int tx = threadIdx.x;
  const int64_t so = (int64_t)s * a.N;
  const T *cb = a.cpml + (int64_t)s * a.cstride;
  const AxisCoef<T> cx = axis_coef(cb, h, 0), cz = axis_coef(cb, h, 1);

  __shared__ T rvx[4][TXM + 6];   // vx^{it-1} rows (slot j&3), x in [I0-3, I0+TXM+3)
  __shared__ T rvz[5][TXM + 3];   // vz^{it-1} rows (slot j%5), x in [I0-1, I0+TXM+2)
  __shared__ T rp[5][TXM + 3];    // p^{it} rows (slot j%5),    x in [I0-1, I0+TXM+2)
  __shared__ int s_pts[2];
  if (tx == 0) {
    const int *sr = a.pt.srow + (int64_t)s * (a.pt.nrows + 1);
    const int *rr = a.pt.rrow + (int64_t)s * (a.pt.nrows + 1);
    s_pts[0] = sr[max(Z0 - 1, 0)] < sr[min(Z1 + 2, nz)];
    s_pts[1] = a.traces != nullptr && rr[Z0] < rr[Z1];
  }

  // column duties: own column gi; halo columns of vx (6), of vz / p / m0 (3)
  const int gi = I0 + tx;
  const int hvx_lx = tx < 3 ? tx : TXM + tx;                 // tx < 6
  const int hp_lx = tx == 0 ? 0 : TXM + tx;                   // tx < 3
  const int hvx_x = I0 - 3 + hvx_lx, hp_x = I0 - 1 + hp_lx;
  auto ld_vx = [&](int x, int j) -> T {
    return (x >= 0 && x <= nx - 2 && j >= 0 && j <= nz - 1) ? a.vx_o[so + (int64_t)j * nx + x] : T(0);
  };
  auto ld_vz = [&](int x, int j) -> T {
    return (x >= 0 && x <= nx - 1 && j >= 0 && j <= nz - 2) ? a.vz_o[so + (int64_t)j * nx + x] : T(0);
  };
  auto ld_f = [&](const T *f, int64_t off, int x, int j) -> T {
    return (x >= 0 && x <= nx - 1 && j >= 0 && j <= nz - 1) ? f[off + (int64_t)j * nx + x] : T(0);
  };
  auto rz5 = [](int j) { return (j + 10) % 5; };

  // vz rows Z0-3 .. Z0-1 straight into the ring
  for (int j = Z0 - 3; j <= Z0 - 1; j++) {
    rvz[rz5(j)][tx + 1] = ld_vz(gi, j);
    if (tx < 3) rvz[rz5(j)][hp_lx] = ld_vz(hp_x, j);
  }
  // registers for row j: vx(j), vz(j+1), p(j), m0(j) with halos; m1x, m1z(j-2)
  T n_vx, n_vxh = 0, n_vz, n_vzh = 0, n_p, n_ph = 0, n_m0, n_m0h = 0, n_m1x, n_m1z;
  auto issue = [&](int j) {
    n_vx = ld_vx(gi, j);
    n_vz = ld_vz(gi, j + 1);
    n_p = ld_f(a.p_o, so, gi, j);
    n_m0 = ld_f(a.m0, 0, gi, j);
    n_m1x = (gi <= nx - 2 && j - 2 >= 0 && j - 2 <= nz - 1) ? a.m1x[(int64_t)(j - 2) * nx + gi] : T(0);
    n_m1z = (gi <= nx - 1 && j - 2 >= 0 && j - 2 <= nz - 2) ? a.m1z[(int64_t)(j - 2) * nx + gi] : T(0);
    if (tx < 6) n_vxh = ld_vx(hvx_x, j);
    if (tx < 3) {
      n_vzh = ld_vz(hp_x, j + 1);
      n_ph = ld_f(a.p_o, so, hp_x, j);
      n_m0h = ld_f(a.m0, 0, hp_x, j);
    }
  };
  issue(Z0 - 1);
  __syncthreads();
  const bool any_src = s_pts[0] != 0, any_rec = s_pts[1] != 0;
  const int sb = store_base(a.smode, a.it, nts, a.S, a.cbase);

  // new pressure at row j, LDS column lx (x = I0-1+lx)
  auto new_p = [&](int lx, int j, T pold, T m0v, bool owned) -> T {
    const int x = I0 - 1 + lx;
    if (x < 0 || x >= nx || j < 0 || j >= nz) return T(0);
    const int64_t c = (int64_t)j * nx + x;
    T pv = pold;
    if (x >= 1 && x <= nx - 2 && j >= 1 && j <= nz - 2) {
      const T *vr = rvx[(j + 4) & 3];
      T dvx = d4(vr[lx], vr[lx + 1], vr[lx + 2], vr[lx + 3]) * a.idx;
      if (x <= h || x >= nx - h - 1) {
        const int k = x <= h ? x : x - nx + 2 * h + 2;
        const int64_t qx = (int64_t)s * a.sxx + (int64_t)j * (2 * h + 2) + k;
        const T xi = cx.b(k) * a.xix_o[qx] + cx.a(k) * dvx;
        if (owned) a.xix_n[qx] = xi;
        dvx = dvx + xi;
      }
      T dvz = d4(rvz[rz5(j - 2)][lx], rvz[rz5(j - 1)][lx], rvz[rz5(j)][lx], rvz[rz5(j + 1)][lx]) * a.idz;
      if (j <= h || j >= nz - h - 1) {
        const int k = j <= h ? j : j - nz + 2 * h + 2;
        const int64_t qz = (int64_t)s * a.sxz + (int64_t)k * nx + x;
        const T xi = cz.b(k) * a.xiz_o[qz] + cz.a(k) * dvz;
        if (owned) a.xiz_n[qz] = xi;
        dvz = dvz + xi;
      }
      pv = pv - m0v * (dvx + dvz);
    }
    const int u = any_src ? find_point(a.pt.srow, a.pt.usrc_cell, a.pt.nrows, s, j, c) : -1;
    if (u >= 0) {
      const T *tf = a.srctf + a.pt.off_tf[s] + (a.it - 1);
      for (int k = a.pt.usrc_ptr[u]; k < a.pt.usrc_ptr[u + 1]; k++) pv += tf[(int64_t)nts * a.pt.usrc_list[k]];
    }
    if (owned) {
      st_nt(a.p_n + so + c, pv);
      if (sb >= 0) {
        st_nt(a.pbuf + (int64_t)(a.it - sb) * a.pslot + so + c, pv);
        if (a.smode == 1 && a.it == sb + 1) st_nt(a.pbuf + so + c, pold);
      }
      if (any_rec) {
        const int r = find_point(a.pt.rrow, a.pt.urec_cell, a.pt.nrows, s, j, c);
        if (r >= 0) {
          T *tr = a.traces + a.pt.off_tr[s] + (a.it - 1);
          for (int k = a.pt.urec_ptr[r]; k < a.pt.urec_ptr[r + 1]; k++) tr[(int64_t)nts * a.pt.urec_list[k]] = pv;
        }
      }
    }
    return pv;
  };

  for (int j = Z0 - 1; j <= Z1 + 1; j++) {
    // commit row j's loads to the rings and registers
    rvx[(j + 4) & 3][tx + 3] = n_vx;
    rvz[rz5(j + 1)][tx + 1] = n_vz;
    if (tx < 6) rvx[(j + 4) & 3][hvx_lx] = n_vxh;
    if (tx < 3) rvz[rz5(j + 1)][hp_lx] = n_vzh;
    const T c_p = n_p, c_ph = n_ph, c_m0 = n_m0, c_m0h = n_m0h, c_m1x = n_m1x, c_m1z = n_m1z;
    if (j + 1 <= Z1 + 1) issue(j + 1);
    __syncthreads();
    // pressure of row j (owned rows write HBM)
    const bool own_row = j >= Z0 && j < Z1;
    rp[rz5(j)][tx + 1] = new_p(tx + 1, j, c_p, c_m0, own_row && gi < nx);
    if (tx < 3) rp[rz5(j)][hp_lx] = new_p(hp_lx, j, c_ph, c_m0h, false);
    __syncthreads();
    // velocities of row jv = j-2 (update_vx_CPML! / update_vy_CPML!, :39-75)
    const int jv = j - 2;
    if (jv >= Z0 && jv < Z1 && gi < nx) {
      const int64_t c = (int64_t)jv * nx + gi;
      if (gi <= nx - 2) {
        const T *pr = rp[rz5(jv)];
        T d = d4(pr[tx], pr[tx + 1], pr[tx + 2], pr[tx + 3]) * a.idx;
        if (gi <= h - 1 || gi >= nx - h - 1) {
          const int k = gi <= h - 1 ? gi : gi + 1 - nx + 2 * h;
          const int64_t q = (int64_t)s * a.spx + (int64_t)jv * (2 * h) + k;
          const T ps = cx.bh(k) * a.psx_o[q] + cx.ah(k) * d;
          a.psx_n[q] = ps;
          d = d + ps;
        }
        a.vx_n[so + c] = rvx[(jv + 4) & 3][tx + 3] - c_m1x * d;
      }
      if (jv <= nz - 2) {
        T d = d4(rp[rz5(jv - 1)][tx + 1], rp[rz5(jv)][tx + 1], rp[rz5(jv + 1)][tx + 1], rp[rz5(jv + 2)][tx + 1]) *
              a.idz;
        if (jv <= h - 1 || jv >= nz - h - 1) {
          const int k = jv <= h - 1 ? jv : jv + 1 - nz + 2 * h;
          const int64_t q = (int64_t)s * a.spz + (int64_t)k * nx + gi;
          const T ps = cz.bh(k) * a.psz_o[q] + cz.ah(k) * d;
          a.psz_n[q] = ps;
          d = d + ps;
        }
        a.vz_n[so + c] = rvz[rz5(jv)][tx + 1] - c_m1z * d;
      }
    }
  }
}

// Is tile (I0, J0) of shot s an interior tile of the adjoint step: every
// cell the tile step reads or updates (old adjoint pressure three cells out,
// velocities two out, replayed pressure one/two out) is inside the grid and
// outside the C-PML strips, and no receiver lies in its rows?
template <int TZ, typename T>
__device__ __forceinline__ bool vd2d_adj_is_lean(const Vd2dArgs<T> &a, int s, int I0, int J0) {
  const int nx = a.nx, nz = a.nz, h = a.h;
  if (!(I0 - 3 > h && I0 + TX + 3 < nx - h - 1 && J0 - 3 > h && J0 + TZ + 3 < nz - h - 1)) return false;
  const int *rr = a.pt.rrow + (int64_t)s * (a.pt.nrows + 1);
  return rr[J0] == rr[J0 + TZ];
}

// Adjoint step of an interior tile (vd2d_adj_is_lean): the updates and
// correlations of vd2d_adj_kernel, in the same operand order, without
// per-cell tests.
template <typename T, int TZ>
struct AdjTileModel {
  static constexpr int R = TZ / BY, HR = (3 * TZ + 3 * TX + NT - 1) / NT;
  T m1x[R], m1z[R], m0[R], hm[HR];
};

// Model factors an interior adjoint tile reads (the same for every shot):
// m1x, m1z, m0 on the thread's tile cells; m1x on the v~x halo columns
// I0-2, I0-1, I0+TX and m1z on the v~z halo rows J0-2, J0-1, J0+TZ.
template <typename T, int TZ>
__device__ __forceinline__ void vd2d_adj_lean_model(const Vd2dArgs<T> &a, int I0, int J0, AdjTileModel<T, TZ> &m) {
  constexpr int R = TZ / BY, HX = 3 * TZ, H = HX + 3 * TX, HR = AdjTileModel<T, TZ>::HR;
  const int nx = a.nx;
  const int tx = threadIdx.x, ty = threadIdx.y, tid = ty * TX + tx;
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int c = (J0 + ty + BY * r) * nx + I0 + tx;
    m.m1x[r] = a.m1x[c];
    m.m1z[r] = a.m1z[c];
    m.m0[r] = a.m0[c];
  }
#pragma unroll
  for (int k = 0; k < HR; k++) {
    const int q = tid + k * NT;
    T v = 0;
    if (q < HX) {
      const int col = q / TZ, lz = q % TZ;
      v = a.m1x[(J0 + lz) * nx + I0 - 2 + (col < 2 ? col : TX + 2)];
    } else if (q < H) {
      const int row = (q - HX) / TX, lx = (q - HX) % TX;
      v = a.m1z[(J0 - 2 + (row < 2 ? row : TZ + 2)) * nx + I0 + lx];
    }
    m.hm[k] = v;
  }
}

template <typename T, int TZ>
__device__ __forceinline__ void vd2d_adj_lean_tile(const Vd2dArgs<T> &a, int s, int I0, int J0,
                                                   T (&s_p)[TZ + 6][TX + 6], T (&s_pc)[TZ + 3][TX + 3],
                                                   T (&s_vx)[TZ][TX + 3], T (&s_vz)[TZ + 3][TX],
                                                   const AdjTileModel<T, TZ> &m) {
  constexpr int R = TZ / BY;
  const int nx = a.nx;
  const int tx = threadIdx.x, ty = threadIdx.y, tid = ty * TX + tx;
  const int64_t so = (int64_t)s * a.N;
  const int slot = a.it - a.cbase;
  const T *__restrict__ pc_ = a.pbuf + (int64_t)slot * a.pslot + so;        // p^{it}
  const T *__restrict__ po_ = a.pbuf + (int64_t)(slot - 1) * a.pslot + so;  // p^{it-1}
  const T *__restrict__ pa = a.p_o + so;
  const T *__restrict__ vxo = a.vx_o + so;
  const T *__restrict__ vzo = a.vz_o + so;

  // every global load of the thread is issued before its first LDS store.
  // Old adjoint pressure: full rows on the tile rows (x arm), tile columns
  // on the three rows above and below (z arm); p^{it} alike.
  constexpr int KP = (TZ + 6 + BY - 1) / BY, KC = (TZ + 3 + BY - 1) / BY;
  T lp0[KP], lp1[KP], lc0[KC], lc1[KC];
#pragma unroll
  for (int k = 0; k < KP; k++) {
    const int lz = ty + k * BY;
    const int c = (J0 - 3 + lz) * nx + I0 - 3;
    const bool arm = lz >= 3 && lz < TZ + 3;
    lp0[k] = lz < TZ + 6 ? pa[c + (arm ? 0 : 3) + tx] : T(0);
    lp1[k] = arm && tx < 6 ? pa[c + TX + tx] : T(0);
  }
#pragma unroll
  for (int k = 0; k < KC; k++) {
    const int lz = ty + k * BY;
    const int c = (J0 - 1 + lz) * nx + I0 - 1;
    const bool arm = lz >= 1 && lz < TZ + 1;
    lc0[k] = lz < TZ + 3 ? pc_[c + (arm ? 0 : 1) + tx] : T(0);
    lc1[k] = arm && tx < 3 ? pc_[c + TX + tx] : T(0);
  }
  T rvx[R], rvz[R], rpo[R], rg0[R], rg1x[R], rg1z[R];
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int c = (J0 + ty + BY * r) * nx + I0 + tx;
    rvx[r] = vxo[c];
    rvz[r] = vzo[c];
    rpo[r] = po_[c];
    rg0[r] = a.g0[so + c];
    rg1x[r] = a.g1x[so + c];
    rg1z[r] = a.g1z[so + c];
  }
  // velocity halo: v~x columns I0-2, I0-1, I0+TX on tile rows; v~z rows
  // J0-2, J0-1, J0+TZ on tile columns
  constexpr int HX = 3 * TZ, H = HX + 3 * TX, HR = AdjTileModel<T, TZ>::HR;
  T hv[HR];
#pragma unroll
  for (int k = 0; k < HR; k++) {
    const int q = tid + k * NT;
    T v = 0;
    if (q < HX) {
      const int col = q / TZ, lz = q % TZ;
      v = vxo[(J0 + lz) * nx + I0 - 2 + (col < 2 ? col : TX + 2)];
    } else if (q < H) {
      const int row = (q - HX) / TX, lx = (q - HX) % TX;
      v = vzo[(J0 - 2 + (row < 2 ? row : TZ + 2)) * nx + I0 + lx];
    }
    hv[k] = v;
  }
  const T(&rm1x)[R] = m.m1x;
  const T(&rm1z)[R] = m.m1z;
  const T(&rm0)[R] = m.m0;
  const T(&hm)[HR] = m.hm;
#pragma unroll
  for (int k = 0; k < KP; k++) {
    const int lz = ty + k * BY;
    if (lz >= 3 && lz < TZ + 3) {
      s_p[lz][tx] = lp0[k];
      if (tx < 6) s_p[lz][TX + tx] = lp1[k];
    } else if (lz < TZ + 6) {
      s_p[lz][tx + 3] = lp0[k];
    }
  }
#pragma unroll
  for (int k = 0; k < KC; k++) {
    const int lz = ty + k * BY;
    if (lz >= 1 && lz < TZ + 1) {
      s_pc[lz][tx] = lc0[k];
      if (tx < 3) s_pc[lz][TX + tx] = lc1[k];
    } else if (lz < TZ + 3) {
      s_pc[lz][tx + 1] = lc0[k];
    }
  }
  __syncthreads();

  auto new_vx = [&](int lx, int lz, T vold, T m1) -> T {
    const T d = d4(s_p[lz + 3][lx], s_p[lz + 3][lx + 1], s_p[lz + 3][lx + 2], s_p[lz + 3][lx + 3]) * a.idx;
    return vold - m1 * d;
  };
  auto new_vz = [&](int lx, int lz, T vold, T m1) -> T {
    const T d = d4(s_p[lz][lx + 3], s_p[lz + 1][lx + 3], s_p[lz + 2][lx + 3], s_p[lz + 3][lx + 3]) * a.idz;
    return vold - m1 * d;
  };
  T *__restrict__ vxn = a.vx_n + so;
  T *__restrict__ vzn = a.vz_n + so;
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int lz = ty + BY * r;
    const int c = (J0 + lz) * nx + I0 + tx;
    const T vx = new_vx(tx + 2, lz, rvx[r], rm1x[r]);
    const T vz = new_vz(tx, lz + 2, rvz[r], rm1z[r]);
    st_nt(vxn + c, vx);
    st_nt(vzn + c, vz);
    s_vx[lz][tx + 2] = vx;
    s_vz[lz + 2][tx] = vz;
  }
#pragma unroll
  for (int k = 0; k < HR; k++) {
    const int q = tid + k * NT;
    if (q < HX) {
      const int col = q / TZ, lz = q % TZ;
      const int lx = col < 2 ? col : TX + 2;
      s_vx[lz][lx] = new_vx(lx, lz, hv[k], hm[k]);
    } else if (q < H) {
      const int row = (q - HX) / TX, lx = (q - HX) % TX;
      const int lz = row < 2 ? row : TZ + 2;
      s_vz[lz][lx] = new_vz(lx, lz, hv[k], hm[k]);
    }
  }
  __syncthreads();

  T *__restrict__ pn = a.p_n + so;
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int lz = ty + BY * r;
    const int c = (J0 + lz) * nx + I0 + tx;
    T pv = s_p[lz + 3][tx + 3];
    const T dvx = d4(s_vx[lz][tx], s_vx[lz][tx + 1], s_vx[lz][tx + 2], s_vx[lz][tx + 3]) * a.idx;
    const T dvz = d4(s_vz[lz][tx], s_vz[lz + 1][tx], s_vz[lz + 2][tx], s_vz[lz + 3][tx]) * a.idz;
    pv = pv - rm0[r] * (dvx + dvz);
    st_nt(pn + c, pv);
    const T pcv = s_pc[lz + 1][tx + 1];
    const T g0 = rg0[r] - (pv * (pcv - rpo[r]) * a.idt);
    st_nt(a.g0 + so + c, g0);
    const T dpx = d4(s_pc[lz + 1][tx], pcv, s_pc[lz + 1][tx + 2], s_pc[lz + 1][tx + 3]) * a.idx;
    const T g1x = rg1x[r] + s_vx[lz][tx + 2] * dpx;
    st_nt(a.g1x + so + c, g1x);
    const T dpz = d4(s_pc[lz][tx + 1], pcv, s_pc[lz + 2][tx + 1], s_pc[lz + 3][tx + 1]) * a.idz;
    const T g1z = rg1z[r] + s_vz[lz + 2][tx] * dpz;
    st_nt(a.g1z + so + c, g1z);
  }
}

// Interior tiles of an adjoint step; blocks of other tiles return at once
// and vd2d_adj_kernel<T, TZ, false>, launched right after on the same grid,
// steps them.
template <typename T, int TZ>
__global__ __launch_bounds__(NT) void vd2d_adj_lean(Vd2dArgs<T> a) {
  int bx, bz, s;
  vd2d_tile_of(a, xcd_tile(blockIdx.x, gridDim.x), bx, bz, s);
  const int nts = a.nt_shot[s];
  if (a.it > nts) return;
  const int I0 = bx * TX, J0 = bz * TZ;
  if (!vd2d_adj_is_lean<TZ>(a, s, I0, J0)) return;
  __shared__ T s_p[TZ + 6][TX + 6];   // p~^{old}: x in [I0-3, I0+TX+3), z in [J0-3, J0+TZ+3) (cross)
  __shared__ T s_pc[TZ + 3][TX + 3];  // p^{it}:   x in [I0-1, I0+TX+2), z in [J0-1, J0+TZ+2) (cross)
  __shared__ T s_vx[TZ][TX + 3];      // v~x^{new}: x in [I0-2, I0+TX+1), z in [J0, J0+TZ)
  __shared__ T s_vz[TZ + 3][TX];      // v~z^{new}: x in [I0, I0+TX), z in [J0-2, J0+TZ+1)
  AdjTileModel<T, TZ> m;
  vd2d_adj_lean_model<T, TZ>(a, I0, J0, m);
  vd2d_adj_lean_tile<T, TZ>(a, s, I0, J0, s_p, s_pc, s_vx, s_vz, m);
}

// Adjoint step of a tile that is not interior: the general path with
// per-cell tests (C-PML memory variables, edges, residual injection).
template <typename T, int TZ>
__device__ __forceinline__ void vd2d_adj_general_tile(const Vd2dArgs<T> &a, int s, int nts, int I0, int J0,
                                                      T (&s_p)[TZ + 6][TX + 6], T (&s_pc)[TZ + 3][TX + 3],
                                                      T (&s_vx)[TZ][TX + 3], T (&s_vz)[TZ + 3][TX]) {
  constexpr int R = TZ / BY;
  const int nx = a.nx, nz = a.nz, h = a.h;
  const int tx = threadIdx.x, ty = threadIdx.y, tid = ty * TX + tx;
  const int64_t so = (int64_t)s * a.N;
  const T *cb = a.cpml + (int64_t)s * a.cstride;
  const AxisCoef<T> cx = axis_coef(cb, h, 0), cz = axis_coef(cb, h, 1);
  const int slot = a.it - a.cbase;
  const T *pc_ = a.pbuf + (int64_t)slot * a.pslot + so;        // p^{it}
  const T *po_ = a.pbuf + (int64_t)(slot - 1) * a.pslot + so;  // p^{it-1}

  // ---- phase 0: all global loads issued before the first LDS store ----------
  constexpr int QP = (TZ + 6) * (TX + 6), KQP = (QP + NT - 1) / NT;
  constexpr int QC = (TZ + 3) * (TX + 3), KQC = (QC + NT - 1) / NT;
  T gp[KQP], gc[KQC];
#pragma unroll
  for (int k = 0; k < KQP; k++) {
    const int q = tid + k * NT;
    const int lz = q / (TX + 6), lx = q % (TX + 6);
    const bool xarm = lz >= 3 && lz < TZ + 3, zarm = lx >= 3 && lx < TX + 3;
    const int gi = I0 - 3 + lx, gj = J0 - 3 + lz;
    T v = 0;
    if (q < QP && (xarm || zarm) && gi >= 0 && gi <= nx - 1 && gj >= 0 && gj <= nz - 1)
      v = a.p_o[so + (int64_t)gj * nx + gi];
    gp[k] = v;
  }
#pragma unroll
  for (int k = 0; k < KQC; k++) {
    const int q = tid + k * NT;
    const int lz = q / (TX + 3), lx = q % (TX + 3);
    const bool xarm = lz >= 1 && lz <= TZ, zarm = lx >= 1 && lx <= TX;
    const int gi = I0 - 1 + lx, gj = J0 - 1 + lz;
    T v = 0;
    if (q < QC && (xarm || zarm) && gi >= 0 && gi <= nx - 1 && gj >= 0 && gj <= nz - 1)
      v = pc_[(int64_t)gj * nx + gi];
    gc[k] = v;
  }
  const int gi = I0 + tx;
  T rvx[R], rvz[R], rm1x[R], rm1z[R], rm0[R], rpo[R], rg0[R], rg1x[R], rg1z[R];
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int gj = J0 + ty + BY * r;
    const bool ok = gi < nx && gj < nz;
    const int64_t c = (int64_t)gj * nx + gi;
    rvx[r] = ok ? a.vx_o[so + c] : T(0);
    rvz[r] = ok ? a.vz_o[so + c] : T(0);
    rm1x[r] = ok ? a.m1x[c] : T(0);
    rm1z[r] = ok ? a.m1z[c] : T(0);
    rm0[r] = ok ? a.m0[c] : T(0);
    rpo[r] = ok ? po_[c] : T(0);
    rg0[r] = ok ? a.g0[so + c] : T(0);
    rg1x[r] = ok ? a.g1x[so + c] : T(0);
    rg1z[r] = ok ? a.g1z[so + c] : T(0);
  }
  // velocity halo: v~x columns I0-2, I0-1, I0+TX on tile rows; v~z rows
  // J0-2, J0-1, J0+TZ on tile columns
  constexpr int HX = 3 * TZ, H = HX + 3 * TX, HR = (H + NT - 1) / NT;
  __shared__ int s_rec;
  if (tid == 0) {
    const int *rr = a.pt.rrow + (int64_t)s * (a.pt.nrows + 1);
    s_rec = rr[J0] < rr[min(J0 + TZ, nz)];
  }
  T hv[HR], hm[HR];
  int hq[HR];
#pragma unroll
  for (int k = 0; k < HR; k++) {
    const int q = tid + k * NT;
    T v = 0, m = 0;
    if (q < HX) {
      const int col = q / TZ, lz = q % TZ;
      const int lx = col < 2 ? col : TX + 2;
      const int gi2 = I0 - 2 + lx, gj2 = J0 + lz;
      if (gi2 >= 0 && gi2 <= nx - 2 && gj2 <= nz - 1) {
        const int64_t c2 = (int64_t)gj2 * nx + gi2;
        v = a.vx_o[so + c2];
        m = a.m1x[c2];
      }
    } else if (q < H) {
      const int row = (q - HX) / TX, lx = (q - HX) % TX;
      const int lz = row < 2 ? row : TZ + 2;
      const int gi2 = I0 + lx, gj2 = J0 - 2 + lz;
      if (gi2 <= nx - 1 && gj2 >= 0 && gj2 <= nz - 2) {
        const int64_t c2 = (int64_t)gj2 * nx + gi2;
        v = a.vz_o[so + c2];
        m = a.m1z[c2];
      }
    }
    hq[k] = q;
    hv[k] = v;
    hm[k] = m;
  }
#pragma unroll
  for (int k = 0; k < KQP; k++) {
    const int q = tid + k * NT;
    if (q < QP) s_p[q / (TX + 6)][q % (TX + 6)] = gp[k];
  }
#pragma unroll
  for (int k = 0; k < KQC; k++) {
    const int q = tid + k * NT;
    if (q < QC) s_pc[q / (TX + 3)][q % (TX + 3)] = gc[k];
  }
  __syncthreads();

  // ---- phase 1: velocities first (adjoint_onestep_CPML!, :163-171) --------
  auto new_vx = [&](int lx, int lz, T vold, T m1, bool owned) -> T {
    const int gi2 = I0 - 2 + lx, gj2 = J0 + lz;
    if (gi2 < 0 || gi2 > nx - 2 || gj2 > nz - 1) return T(0);
    T d = d4(s_p[lz + 3][lx], s_p[lz + 3][lx + 1], s_p[lz + 3][lx + 2], s_p[lz + 3][lx + 3]) * a.idx;
    if (gi2 <= h - 1 || gi2 >= nx - h - 1) {
      const int k = gi2 <= h - 1 ? gi2 : gi2 + 1 - nx + 2 * h;
      const int64_t qq = (int64_t)s * a.spx + (int64_t)gj2 * (2 * h) + k;
      const T ps = cx.bh(k) * a.psx_o[qq] + cx.ah(k) * d;
      if (owned) a.psx_n[qq] = ps;
      d = d + ps;
    }
    const T v = vold - m1 * d;
    if (owned) st_nt(a.vx_n + so + (int64_t)gj2 * nx + gi2, v);
    return v;
  };
  auto new_vz = [&](int lx, int lz, T vold, T m1, bool owned) -> T {
    const int gi2 = I0 + lx, gj2 = J0 - 2 + lz;
    if (gi2 > nx - 1 || gj2 < 0 || gj2 > nz - 2) return T(0);
    T d = d4(s_p[lz][lx + 3], s_p[lz + 1][lx + 3], s_p[lz + 2][lx + 3], s_p[lz + 3][lx + 3]) * a.idz;
    if (gj2 <= h - 1 || gj2 >= nz - h - 1) {
      const int k = gj2 <= h - 1 ? gj2 : gj2 + 1 - nz + 2 * h;
      const int64_t qq = (int64_t)s * a.spz + (int64_t)k * nx + gi2;
      const T ps = cz.bh(k) * a.psz_o[qq] + cz.ah(k) * d;
      if (owned) a.psz_n[qq] = ps;
      d = d + ps;
    }
    const T v = vold - m1 * d;
    if (owned) st_nt(a.vz_n + so + (int64_t)gj2 * nx + gi2, v);
    return v;
  };
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int lz = ty + BY * r;
    s_vx[lz][tx + 2] = new_vx(tx + 2, lz, rvx[r], rm1x[r], true);
    s_vz[lz + 2][tx] = new_vz(tx, lz + 2, rvz[r], rm1z[r], true);
  }
#pragma unroll
  for (int k = 0; k < HR; k++) {
    const int q = hq[k];
    if (q < HX) {
      const int col = q / TZ, lz = q % TZ;
      const int lx = col < 2 ? col : TX + 2;
      s_vx[lz][lx] = new_vx(lx, lz, hv[k], hm[k], false);
    } else if (q < H) {
      const int row = (q - HX) / TX, lx = (q - HX) % TX;
      const int lz = row < 2 ? row : TZ + 2;
      s_vz[lz][lx] = new_vz(lx, lz, hv[k], hm[k], false);
    }
  }
  __syncthreads();

  // ---- phase 2: pressure (update_p_CPML!), residual injection, correlation
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int lz = ty + BY * r;
    const int gj = J0 + lz;
    if (gi >= nx || gj >= nz) continue;
    const int64_t c = (int64_t)gj * nx + gi;
    T pv = s_p[lz + 3][tx + 3];
    if (gi >= 1 && gi <= nx - 2 && gj >= 1 && gj <= nz - 2) {
      T dvx = d4(s_vx[lz][tx], s_vx[lz][tx + 1], s_vx[lz][tx + 2], s_vx[lz][tx + 3]) * a.idx;
      if (gi <= h || gi >= nx - h - 1) {
        const int k = gi <= h ? gi : gi - nx + 2 * h + 2;
        const int64_t qx = (int64_t)s * a.sxx + (int64_t)gj * (2 * h + 2) + k;
        const T xi = cx.b(k) * a.xix_o[qx] + cx.a(k) * dvx;
        a.xix_n[qx] = xi;
        dvx = dvx + xi;
      }
      T dvz = d4(s_vz[lz][tx], s_vz[lz + 1][tx], s_vz[lz + 2][tx], s_vz[lz + 3][tx]) * a.idz;
      if (gj <= h || gj >= nz - h - 1) {
        const int k = gj <= h ? gj : gj - nz + 2 * h + 2;
        const int64_t qz = (int64_t)s * a.sxz + (int64_t)k * nx + gi;
        const T xi = cz.b(k) * a.xiz_o[qz] + cz.a(k) * dvz;
        a.xiz_n[qz] = xi;
        dvz = dvz + xi;
      }
      pv = pv - rm0[r] * (dvx + dvz);
    }
    // residual injection with prescale_residuals! by fact_m0 (:77-89)
    const int u = s_rec ? find_point(a.pt.rrow, a.pt.urec_cell, a.pt.nrows, s, gj, c) : -1;
    if (u >= 0) {
      const T *rs = a.res + a.pt.off_tr[s] + (a.it - 1);
      for (int k = a.pt.urec_ptr[u]; k < a.pt.urec_ptr[u + 1]; k++)
        pv += rs[(int64_t)nts * a.pt.urec_list[k]] * rm0[r];
    }
    st_nt(a.p_n + so + c, pv);
    // correlate_gradient_m0! (correlate_gradient_xPU.jl:12-21)
    const T pcv = s_pc[lz + 1][tx + 1];
    st_nt(a.g0 + so + c, rg0[r] - (pv * (pcv - rpo[r]) * a.idt));
    // correlate_gradient_m1! (acoustic2D_VD_xPU.jl:180-198), 4th order, no C-PML
    if (gi <= nx - 2) {
      const T dpx = d4(s_pc[lz + 1][tx], pcv, s_pc[lz + 1][tx + 2], s_pc[lz + 1][tx + 3]) * a.idx;
      st_nt(a.g1x + so + c, rg1x[r] + s_vx[lz][tx + 2] * dpx);
    }
    if (gj <= nz - 2) {
      const T dpz = d4(s_pc[lz][tx + 1], pcv, s_pc[lz + 2][tx + 1], s_pc[lz + 3][tx + 1]) * a.idz;
      st_nt(a.g1z + so + c, rg1z[r] + s_vz[lz + 2][tx] * dpz);
    }
  }
}

// Adjoint step it: (p~, v~)^{it+1} -> (p~, v~)^{it}, then the correlation
// with p^{it}, p^{it-1} of the replayed segment.  Interior tiles are stepped
// inline (FOLD, one launch per step) or left to vd2d_adj_lean.
template <typename T, int TZ, bool FOLD>
__global__ __launch_bounds__(NT) void vd2d_adj_kernel(Vd2dArgs<T> a) {
  int bx, bz, s;
  vd2d_tile_of(a, xcd_tile(blockIdx.x, gridDim.x), bx, bz, s);
  const int nts = a.nt_shot[s];
  if (a.it > nts) return;
  const int I0 = bx * TX, J0 = bz * TZ;
  __shared__ T s_p[TZ + 6][TX + 6];   // p~^{old}: x in [I0-3, I0+TX+3), z in [J0-3, J0+TZ+3) (cross)
  __shared__ T s_pc[TZ + 3][TX + 3];  // p^{it}:   x in [I0-1, I0+TX+2), z in [J0-1, J0+TZ+2) (cross)
  __shared__ T s_vx[TZ][TX + 3];      // v~x^{new}: x in [I0-2, I0+TX+1), z in [J0, J0+TZ)
  __shared__ T s_vz[TZ + 3][TX];      // v~z^{new}: x in [I0, I0+TX), z in [J0-2, J0+TZ+1)
  if (vd2d_adj_is_lean<TZ>(a, s, I0, J0)) {
    if (FOLD) {
      AdjTileModel<T, TZ> m;
      vd2d_adj_lean_model<T, TZ>(a, I0, J0, m);
      vd2d_adj_lean_tile<T, TZ>(a, s, I0, J0, s_p, s_pc, s_vx, s_vz, m);
    }
    return;
  }
  vd2d_adj_general_tile<T, TZ>(a, s, nts, I0, J0, s_p, s_pc, s_vx, s_vz);
}

// Adjoint step of a pair of shots (2k, 2k+1) per block: the model factors
// of an interior tile are read once for both shots; each shot is stepped
// with the expressions of vd2d_adj_kernel (bitwise the same results).
template <typename T, int TZ>
__global__ __launch_bounds__(NT) void vd2d_adj_pair_kernel(Vd2dArgs<T> a) {
  const int b = xcd_tile(blockIdx.x, gridDim.x);
  const int bx = b % a.nbx, bzs = b / a.nbx, bz = bzs % a.nbz, pr = bzs / a.nbz;
  const int I0 = bx * TX, J0 = bz * TZ;
  __shared__ T s_p[TZ + 6][TX + 6];
  __shared__ T s_pc[TZ + 3][TX + 3];
  __shared__ T s_vx[TZ][TX + 3];
  __shared__ T s_vz[TZ + 3][TX];
  AdjTileModel<T, TZ> m;
  bool have_m = false;
  for (int k = 0; k < 2; k++) {
    const int s = 2 * pr + k;
    if (s >= a.nsh) break;
    const int nts = a.nt_shot[s];
    if (a.it > nts) continue;
    if (k == 1) __syncthreads();   // the LDS tiles of the first shot are consumed
    if (vd2d_adj_is_lean<TZ>(a, s, I0, J0)) {
      if (!have_m) {
        vd2d_adj_lean_model<T, TZ>(a, I0, J0, m);
        have_m = true;
      }
      vd2d_adj_lean_tile<T, TZ>(a, s, I0, J0, s_p, s_pc, s_vx, s_vz, m);
    } else {
      vd2d_adj_general_tile<T, TZ>(a, s, nts, I0, J0, s_p, s_pc, s_vx, s_vz);
    }
  }
}


// Adjoint step marching down z (same strip/chunk decomposition as
// vd2d_fwd_march).  At row j: the new adjoint velocities of row j (vx also
// on the two-left / one-right halo columns) from the ring of old adjoint
// pressure rows j-1..j+2, then the pressure of row j-1 from the rings of new
// velocities, residual injection and the correlation with the replayed
// p^{it} rows j-2..j+1 and p^{it-1}.  Rings are deep enough for two barriers
// per row.
template <typename T, int W>
__global__ __launch_bounds__(64 * W) void vd2d_adj_march(Vd2dArgs<T> a) {
  constexpr int TXM = 64 * W;
  const int b = xcd_tile(blockIdx.x, gridDim.x);
  const int bx = b % a.nbx, bzs = b / a.nbx, bz = bzs % a.nbz, s = bzs / a.nbz;
  const int nts = a.nt_shot[s];
  if (a.it > nts) return;
  const int nx = a.nx, nz = a.nz, h = a.h;
  const int I0 = bx * TXM, Z0 = bz * a.ch, Z1 = min(Z0 + a.ch, nz);
  const int tx = threadIdx.x;
  const int64_t so = (int64_t)s * a.N;
  const T *cb = a.cpml + (int64_t)s * a.cstride;
  const AxisCoef<T> cx = axis_coef(cb, h, 0), cz = axis_coef(cb, h, 1);
  const int slot = a.it - a.cbase;
  const T *pc_ = a.pbuf + (int64_t)slot * a.pslot + so;        // p^{it}
  const T *po_ = a.pbuf + (int64_t)(slot - 1) * a.pslot + so;  // p^{it-1}

  __shared__ T rpo[5][TXM + 6];   // old adjoint p rows (slot j%5), x in [I0-3, I0+TXM+3)
  __shared__ T rpc[6][TXM + 3];   // p^{it} rows (slot j%6),        x in [I0-1, I0+TXM+2)
  __shared__ T rvx[3][TXM + 3];   // new adjoint vx rows (slot j%3), x in [I0-2, I0+TXM+1)
  __shared__ T rvz[5][TXM];       // new adjoint vz rows (slot j%5), x in [I0, I0+TXM)
  __shared__ int s_rec;
  if (tx == 0) {
    const int *rr = a.pt.rrow + (int64_t)s * (a.pt.nrows + 1);
    s_rec = rr[Z0] < rr[Z1];
  }
  const int gi = I0 + tx;
  const int ho_lx = tx < 3 ? tx : TXM + tx;   // tx < 6: old-p halo columns (x = I0-3+ho_lx)
  const int hc_lx = tx == 0 ? 0 : TXM + tx;   // tx < 3: p^{it} halo columns (x = I0-1+hc_lx)
  const int hv_lx = tx < 2 ? tx : TXM + 2;    // tx < 3: vx halo columns (x = I0-2+hv_lx)
  const int ho_x = I0 - 3 + ho_lx, hc_x = I0 - 1 + hc_lx, hv_x = I0 - 2 + hv_lx;
  auto r5 = [](int j) { return (j + 10) % 5; };
  auto r6 = [](int j) { return (j + 12) % 6; };
  auto r3 = [](int j) { return (j + 6) % 3; };
  auto ld_p = [&](const T *f, int x, int j) -> T {
    return (x >= 0 && x <= nx - 1 && j >= 0 && j <= nz - 1) ? f[(int64_t)j * nx + x] : T(0);
  };
  auto ld_vx = [&](const T *f, int x, int j) -> T {
    return (x >= 0 && x <= nx - 2 && j >= 0 && j <= nz - 1) ? f[(int64_t)j * nx + x] : T(0);
  };
  auto ld_vz = [&](const T *f, int x, int j) -> T {
    return (x >= 0 && x <= nx - 1 && j >= 0 && j <= nz - 2) ? f[(int64_t)j * nx + x] : T(0);
  };
  const T *pold = a.p_o + so;

  // preload old p rows Z0-3 .. Z0-1 and p^{it} row Z0-1
  for (int j = Z0 - 3; j <= Z0 - 1; j++) {
    rpo[r5(j)][tx + 3] = ld_p(pold, gi, j);
    if (tx < 6) rpo[r5(j)][ho_lx] = ld_p(pold, ho_x, j);
  }
  rpc[r6(Z0 - 1)][tx + 1] = ld_p(pc_, gi, Z0 - 1);
  if (tx < 3) rpc[r6(Z0 - 1)][hc_lx] = ld_p(pc_, hc_x, Z0 - 1);

  // prefetched per row j: old p / p^{it} row j+2; vx, vz, m1x, m1z row j
  // (vx, m1x also on the halo columns); m0, p^{it-1}, grads of row j-1
  T n_po, n_poh = 0, n_pc, n_pch = 0, n_vx, n_vxh = 0, n_m1x, n_m1xh = 0, n_vz, n_m1z;
  T n_m0, n_pm, n_g0, n_g1x, n_g1z;
  auto issue = [&](int j) {
    n_po = ld_p(pold, gi, j + 2);
    n_pc = ld_p(pc_, gi, j + 2);
    n_vx = ld_vx(a.vx_o + so, gi, j);
    n_m1x = ld_vx(a.m1x, gi, j);
    n_vz = ld_vz(a.vz_o + so, gi, j);
    n_m1z = ld_vz(a.m1z, gi, j);
    n_m0 = ld_p(a.m0, gi, j - 1);
    n_pm = ld_p(po_, gi, j - 1);
    n_g0 = ld_p(a.g0 + so, gi, j - 1);
    n_g1x = ld_p(a.g1x + so, gi, j - 1);
    n_g1z = ld_p(a.g1z + so, gi, j - 1);
    if (tx < 6) n_poh = ld_p(pold, ho_x, j + 2);
    if (tx < 3) {
      n_pch = ld_p(pc_, hc_x, j + 2);
      n_vxh = ld_vx(a.vx_o + so, hv_x, j);
      n_m1xh = ld_vx(a.m1x, hv_x, j);
    }
  };
  issue(Z0 - 2);
  __syncthreads();

  // new adjoint vx at row j, ring column lx (x = I0-2+lx)
  auto new_vx = [&](int lx, int j, T vold, T m1, bool owned) -> T {
    const int x = I0 - 2 + lx;
    if (x < 0 || x > nx - 2 || j < 0 || j > nz - 1) return T(0);
    const T *pr = rpo[r5(j)];
    T d = d4(pr[lx], pr[lx + 1], pr[lx + 2], pr[lx + 3]) * a.idx;
    if (x <= h - 1 || x >= nx - h - 1) {
      const int k = x <= h - 1 ? x : x + 1 - nx + 2 * h;
      const int64_t qq = (int64_t)s * a.spx + (int64_t)j * (2 * h) + k;
      const T ps = cx.bh(k) * a.psx_o[qq] + cx.ah(k) * d;
      if (owned) a.psx_n[qq] = ps;
      d = d + ps;
    }
    const T v = vold - m1 * d;
    if (owned) a.vx_n[so + (int64_t)j * nx + x] = v;
    return v;
  };

  for (int j = Z0 - 2; j <= Z1; j++) {
    rpo[r5(j + 2)][tx + 3] = n_po;
    rpc[r6(j + 2)][tx + 1] = n_pc;
    if (tx < 6) rpo[r5(j + 2)][ho_lx] = n_poh;
    if (tx < 3) rpc[r6(j + 2)][hc_lx] = n_pch;
    const T c_vx = n_vx, c_vxh = n_vxh, c_m1x = n_m1x, c_m1xh = n_m1xh, c_vz = n_vz, c_m1z = n_m1z;
    const T c_m0 = n_m0, c_pm = n_pm, c_g0 = n_g0, c_g1x = n_g1x, c_g1z = n_g1z;
    if (j + 1 <= Z1) issue(j + 1);
    __syncthreads();
    // ---- velocities of row j (adjoint_onestep_CPML!, :163-171) ----------
    const bool own_row = j >= Z0 && j < Z1;
    rvx[r3(j)][tx + 2] = new_vx(tx + 2, j, c_vx, c_m1x, own_row && gi < nx);
    if (tx < 3) rvx[r3(j)][hv_lx] = new_vx(hv_lx, j, c_vxh, c_m1xh, false);
    {
      T v = 0;
      if (gi <= nx - 1 && j >= 0 && j <= nz - 2) {
        T d = d4(rpo[r5(j - 1)][tx + 3], rpo[r5(j)][tx + 3], rpo[r5(j + 1)][tx + 3], rpo[r5(j + 2)][tx + 3]) *
              a.idz;
        if (j <= h - 1 || j >= nz - h - 1) {
          const int k = j <= h - 1 ? j : j + 1 - nz + 2 * h;
          const int64_t qq = (int64_t)s * a.spz + (int64_t)k * nx + gi;
          const T ps = cz.bh(k) * a.psz_o[qq] + cz.ah(k) * d;
          if (own_row) a.psz_n[qq] = ps;
          d = d + ps;
        }
        v = c_vz - c_m1z * d;
        if (own_row) a.vz_n[so + (int64_t)j * nx + gi] = v;
      }
      rvz[r5(j)][tx] = v;
    }
    __syncthreads();
    // ---- pressure of row jp = j-1, residual injection, correlation -------
    const int jp = j - 1;
    if (jp >= Z0 && jp < Z1 && gi < nx) {
      const int64_t c = (int64_t)jp * nx + gi;
      T pv = rpo[r5(jp)][tx + 3];
      if (gi >= 1 && gi <= nx - 2 && jp >= 1 && jp <= nz - 2) {
        const T *vr = rvx[r3(jp)];
        T dvx = d4(vr[tx], vr[tx + 1], vr[tx + 2], vr[tx + 3]) * a.idx;
        if (gi <= h || gi >= nx - h - 1) {
          const int k = gi <= h ? gi : gi - nx + 2 * h + 2;
          const int64_t qx = (int64_t)s * a.sxx + (int64_t)jp * (2 * h + 2) + k;
          const T xi = cx.b(k) * a.xix_o[qx] + cx.a(k) * dvx;
          a.xix_n[qx] = xi;
          dvx = dvx + xi;
        }
        T dvz = d4(rvz[r5(jp - 2)][tx], rvz[r5(jp - 1)][tx], rvz[r5(jp)][tx], rvz[r5(jp + 1)][tx]) * a.idz;
        if (jp <= h || jp >= nz - h - 1) {
          const int k = jp <= h ? jp : jp - nz + 2 * h + 2;
          const int64_t qz = (int64_t)s * a.sxz + (int64_t)k * nx + gi;
          const T xi = cz.b(k) * a.xiz_o[qz] + cz.a(k) * dvz;
          a.xiz_n[qz] = xi;
          dvz = dvz + xi;
        }
        pv = pv - c_m0 * (dvx + dvz);
      }
      const int u = s_rec ? find_point(a.pt.rrow, a.pt.urec_cell, a.pt.nrows, s, jp, c) : -1;
      if (u >= 0) {
        const T *rs = a.res + a.pt.off_tr[s] + (a.it - 1);
        for (int k = a.pt.urec_ptr[u]; k < a.pt.urec_ptr[u + 1]; k++)
          pv += rs[(int64_t)nts * a.pt.urec_list[k]] * c_m0;
      }
      a.p_n[so + c] = pv;
      const T pcv = rpc[r6(jp)][tx + 1];
      a.g0[so + c] = c_g0 - (pv * (pcv - c_pm) * a.idt);
      if (gi <= nx - 2) {
        const T *cr = rpc[r6(jp)];
        const T dpx = d4(cr[tx], pcv, cr[tx + 2], cr[tx + 3]) * a.idx;
        a.g1x[so + c] = c_g1x + rvx[r3(jp)][tx + 2] * dpx;
      }
      if (jp <= nz - 2) {
        const T dpz = d4(rpc[r6(jp - 1)][tx + 1], pcv, rpc[r6(jp + 1)][tx + 1], rpc[r6(jp + 2)][tx + 1]) * a.idz;
        a.g1z[so + c] = c_g1z + rvz[r5(jp)][tx] * dpz;
      }
    }
  }
}

template <typename T>
class Vd2dEngine final : public Engine {
 public:
  explicit Vd2dEngine(PlanCore &core) : c_(core) {
    const swx_plan_desc &d = c_.d;
    nx_ = (int)d.n[0];
    nz_ = (int)d.n[1];
    h_ = d.halo;
    ns_ = d.max_shots;
    N_ = (int64_t)nx_ * nz_;
    spx_ = (int64_t)2 * h_ * nz_;
    spz_ = (int64_t)nx_ * 2 * h_;
    sxx_ = (int64_t)(2 * h_ + 2) * nz_;
    sxz_ = (int64_t)nx_ * (2 * h_ + 2);
    cstride_ = 2 * (8 * h_ + 4);
    const int64_t e = sizeof(T);
    const int64_t F = ns_ * N_;
    m_.alloc(3 * N_ * e);
    st_[0].alloc(2 * 3 * F * e);  // [parity][p, vx, vz][ns][N]
    st_[1].alloc(2 * ns_ * std::max<int64_t>(spx_ + spz_, 1) * e);
    st_[2].alloc(2 * ns_ * (sxx_ + sxz_) * e);
    cpml_.alloc((int64_t)ns_ * cstride_ * e);
    state_bytes_ = m_.bytes() + st_[0].bytes() + st_[1].bytes() + st_[2].bytes() + cpml_.bytes();
    if (d.gradient) {
      ad_[0].alloc(st_[0].bytes());
      ad_[1].alloc(st_[1].bytes());
      ad_[2].alloc(st_[2].bytes());
      grad_.alloc(3 * F * e);
      gout_.alloc(3 * F * e);
      state_bytes_ += ad_[0].bytes() + ad_[1].bytes() + ad_[2].bytes() + grad_.bytes() + gout_.bytes();
      const int64_t slot = F * e;
      ck_one_ = (3 * N_ + spx_ + spz_ + sxx_ + sxz_) * ns_ * e;
      const int64_t avail = (int64_t)c_.budget - state_bytes_;
      // the replay buffer holds S+1 pressure slots
      S_ = choose_segment(d.nt_max, d.check_freq, slot, ck_one_, avail - slot - 2 * ck_one_);
      // check_freq = 1 keeps every step (no replay); otherwise a checkpoint
      // at every multiple of S, as the reference's LinearCheckpointer
      store_all_ = d.check_freq <= 1 && S_ == d.nt_max;
      K_ = (int)ceil_div(d.nt_max, S_);
      pbuf_.alloc((int64_t)(S_ + 1) * slot);
      nck_ = store_all_ ? 0 : d.nt_max / S_;
      ck_.alloc(std::max<int64_t>(nck_ * ck_one_, 1));
    }
    zero(st_);
  }

  void set_model(int nfields, const void *const *fields) override {
    SWX_REQUIRE(nfields == 3 && fields[0] && fields[1] && fields[2], SWX_EINVAL,
                "acoustic VD expects three model fields (fact_m0, fact_m1_stag x, z)");
    const size_t e = sizeof(T);
    SWX_HIP(hipMemsetAsync(m_.get(), 0, m_.bytes(), c_.stream));
    SWX_HIP(hipMemcpyAsync(M(0), fields[0], N_ * e, hipMemcpyHostToDevice, c_.stream));
    // fact_m1_stag[1] is (nx-1) x nz: pitched into the nx x nz slab
    SWX_HIP(hipMemcpy2DAsync(M(1), nx_ * e, fields[1], (nx_ - 1) * e, (nx_ - 1) * e, nz_, hipMemcpyHostToDevice,
                             c_.stream));
    SWX_HIP(hipMemcpyAsync(M(2), fields[2], (int64_t)nx_ * (nz_ - 1) * e, hipMemcpyHostToDevice, c_.stream));
    SWX_HIP(hipStreamSynchronize(c_.stream));
    model_set_ = true;
  }

  void on_shots_set(int nshots, const swx_shot_desc *shots) override {
    std::vector<T> hc = pack_cpml<T>(nshots, shots, 2, h_);
    SWX_HIP(hipMemcpyAsync(cpml_.get(), hc.data(), hc.size() * sizeof(T), hipMemcpyHostToDevice, c_.stream));
    SWX_HIP(hipStreamSynchronize(c_.stream));
    nsh_ = nshots;
    nt_ = c_.pts.nt;
    ntmax_ = *std::max_element(nt_.begin(), nt_.end());
  }

  void forward(bool save) override {
    SWX_REQUIRE(model_set_, SWX_ESTATE, "swx_set_model must be called before running");
    zero(st_);
    tz_fwd_ = choose_steps("SWX_VD2D_TILE_FWD", false);
    if (!tz_fwd_ && !tile_fwd_) {
      const Vd2dArgs<T> a1 = fwd_args(1, 0, save && c_.d.gradient ? 1 : 0, 0, c_.pts.d_traces.as<T>());
      tile_fwd_ = tune("SWX_VD2D_TILE_FWD",
                       candidates({8, 16, Tiles<T>::fwd_max, 308, 316, 300 + Tiles<T>::fwd_max}),
                       [&](int tz) { launch_fwd(a1, tz); });
    }
    if (!tz_fwd_) tz_fwd_ = tile_fwd_;
    for (int it = 1; it <= ntmax_;) {
      progress("forward step", it, ntmax_);
      // a launch of several steps never steps over a checkpoint or snapshot level
      int n = std::min(steps_per_launch(tz_fwd_), ntmax_ - it + 1);
      if (save && nck_ > 0) n = std::min(n, S_ - (it - 1) % S_);
      if (c_.snap_every > 0) n = std::min(n, c_.snap_every - (it - 1) % c_.snap_every);
      fwd_step(it, n, 0, save && c_.d.gradient ? 1 : 0, 0, c_.pts.d_traces.as<T>());
      it += n;
      const int last = it - 1;
      take_snapshots(c_, *this, last);
      if (save && last % S_ == 0) {
        const int k = last / S_;
        if (k >= 1 && k <= nck_) ckpt_copy(k, last, true);
      }
    }
  }

  void adjoint(bool per_shot) override {
    const int Kmax = (int)ceil_div(ntmax_, S_);
    tz_adj_ = choose_steps("SWX_VD2D_TILE_ADJ", true);
    if (!tz_adj_ && !tile_adj_) {
      // timed on a step every shot takes part in (the shortest shot's last
      // step); the history slots it reads are in range, their contents do
      // not matter, and the adjoint state and gradients are cleared below
      const int itt = *std::min_element(nt_.begin(), nt_.end());
      const Vd2dArgs<T> a1 = adj_args(itt, ((itt - 1) / S_) * S_);
      tile_adj_ = tune("SWX_VD2D_TILE_ADJ", candidates({16, 316}), [&](int tz) { launch_adj(a1, tz); });
    }
    if (!tz_adj_) tz_adj_ = tile_adj_;
    zero(ad_);
    SWX_HIP(hipMemsetAsync(grad_.get(), 0, grad_.bytes(), c_.stream));
    const int64_t F = (int64_t)ns_ * N_;
    for (int k = Kmax - 1; k >= 0; k--) {
      progress("adjoint segment", Kmax - k, Kmax);
      const int cb = k * S_;
      // shots whose checkpoint (k+1)S exists replay segment k (initrecover!/
      // recover!/getsaved, checkpointers.jl:80-105): p^{cb} from checkpoint
      // k, cb+1 .. cb+S-1 recomputed, p^{cb+S} from checkpoint k+1
      const int act = cb + S_ - 1;
      bool need = false;
      for (int s = 0; s < nsh_; s++) need |= !store_all_ && nt_[s] > act;
      if (need) {
        if (k == 0) zero(st_);
        else ckpt_copy(k, cb, false);
        dim3 g((unsigned)std::min<int64_t>(ceil_div(N_, 256), 1024), (unsigned)nsh_);
        copy_active_shots<T><<<g, 256, 0, c_.stream>>>(pbuf_.as<T>(), F3(st_, slot(cb), 0), N_,
                                                       c_.pts.d_nt.as<int>(), act);
        SWX_HIP(hipGetLastError());
        for (int it = cb + 1; it <= cb + S_ - 1;) {
          const int n = std::min(steps_per_launch(tz_fwd_), cb + S_ - it);
          fwd_step(it, n, act, 2, cb, nullptr);
          it += n;
        }
        const T *ck1 = reinterpret_cast<const T *>(ck_.as<char>() + (int64_t)k * ck_one_);
        copy_active_shots<T><<<g, 256, 0, c_.stream>>>(pbuf_.as<T>() + (int64_t)S_ * F, ck1, N_,
                                                       c_.pts.d_nt.as<int>(), act);
        SWX_HIP(hipGetLastError());
      }
      const int top = std::min(cb + S_, ntmax_);
      for (int it = top; it >= cb + 1;) {
        const int n = is_stepn(tz_adj_) ? std::min(steps_per_launch(tz_adj_), it - cb) : 1;
        adj_step(it, n, cb);
        it -= n;
      }
    }
    dim3 g((unsigned)std::min<int64_t>(ceil_div(N_, 256), 4096));
    for (int f = 0; f < 3; f++)
      reduce_shots<T><<<g, 256, 0, c_.stream>>>(gout_.as<T>() + f * F, grad_.as<T>() + f * F, N_, nsh_, T(1),
                                                per_shot ? 1 : 0);
    SWX_HIP(hipGetLastError());
  }

  void copy_grad(void *host, bool per_shot) override {
    // per copy: grad_m0 (nx*nz) | grad_m1 x ((nx-1)*nz) | grad_m1 z (nx*(nz-1))
    const size_t e = sizeof(T);
    const int nc = per_shot ? nsh_ : 1;
    const int64_t F = (int64_t)ns_ * N_;
    const int64_t per = N_ + (int64_t)(nx_ - 1) * nz_ + (int64_t)nx_ * (nz_ - 1);
    char *dst = static_cast<char *>(host);
    for (int s = 0; s < nc; s++) {
      char *o = dst + (size_t)s * per * e;
      const T *b0 = gout_.as<T>() + (int64_t)s * N_;
      SWX_HIP(hipMemcpy(o, b0, N_ * e, hipMemcpyDeviceToHost));
      o += N_ * e;
      SWX_HIP(hipMemcpy2D(o, (nx_ - 1) * e, b0 + F, nx_ * e, (nx_ - 1) * e, nz_, hipMemcpyDeviceToHost));
      o += (size_t)(nx_ - 1) * nz_ * e;
      SWX_HIP(hipMemcpy(o, b0 + 2 * F, (size_t)nx_ * (nz_ - 1) * e, hipMemcpyDeviceToHost));
    }
  }

  int64_t bytes_state() const override { return state_bytes_; }
  int64_t bytes_checkpoints() const override { return ck_.bytes(); }
  int64_t bytes_replay() const override { return pbuf_.bytes(); }
  int segment() const override { return S_; }
  void variants(int32_t v[2]) const override { v[0] = used(tz_fwd_); v[1] = used(tz_adj_); }

  // "pcur" and "vcur" = [vx, vz] (acou_forward.jl:116-120): level it is in
  // parity slot(it) right after its step
  int snap_fields(int it, int s, SnapPiece *out) const override {
    const int64_t e = sizeof(T), so = (int64_t)s * N_;
    out[0] = {F3(st_, slot(it), 0) + so, nx_ * e, nx_ * e, nz_};
    out[1] = {F3(st_, slot(it), 1) + so, (nx_ - 1) * e, nx_ * e, nz_};
    out[2] = {F3(st_, slot(it), 2) + so, nx_ * e, nx_ * e, nz_ - 1};
    return 3;
  }

 private:
  T *M(int f) const { return m_.as<T>() + (int64_t)f * N_; }
  // field f (0 p, 1 vx, 2 vz) of parity par in state block b
  T *F3(const DevBuf *b, int par, int f) const { return b[0].as<T>() + ((int64_t)par * 3 + f) * ns_ * N_; }
  T *PSX(const DevBuf *b, int par) const { return b[1].as<T>() + (int64_t)par * ns_ * (spx_ + spz_); }
  T *PSZ(const DevBuf *b, int par) const { return PSX(b, par) + ns_ * spx_; }
  T *XIX(const DevBuf *b, int par) const { return b[2].as<T>() + (int64_t)par * ns_ * (sxx_ + sxz_); }
  T *XIZ(const DevBuf *b, int par) const { return XIX(b, par) + ns_ * sxx_; }

  void zero(DevBuf *b) {
    for (int k = 0; k < 3; k++) SWX_HIP(hipMemsetAsync(b[k].get(), 0, b[k].bytes(), c_.stream));
    (b == st_ ? flip_ : aflip_) = 0;
  }

  // Forward state buffer (0/1) holding time level k.  Single-step launches
  // read level it-1 and write level it into the other buffer; a two-step
  // launch also writes into the other buffer, so it toggles flip_.
  int slot(int k) const { return ((k % 2) + 2 + flip_) % 2; }
  static bool is_stepn(int code) { return code > 500 && code < 600; }
  static int steps_per_launch(int code) { return is_stepn(code) ? code % 10 : code >= 200 && code < 300 ? 2 : 1; }
  // a 2-D tile code and its shot-group codes (code + 1000 k, groups of 2^k
  // shots, k = 1..3) whose group divides the batch
  std::vector<int> with_groups(int code) const {
    std::vector<int> v = {code};
    const int base = code % 100;
    if (code >= 400 || (code >= 100 && code < 300) || (base != 8 && base != 16 && base != 32)) return v;
    for (int k = 1; k <= 3; k++)
      if (nsh_ % (1 << k) == 0 && nsh_ > (1 << k)) v.push_back(code + 1000 * k);
    return v;
  }

  // A tile code as the batch in hand takes it: a code chosen for another batch
  // may group the shots by a number that does not divide this one, and
  // vd2d_tile_of would then send blocks to a shot beyond it.
  int used(int code) const { return nsh_ % (1 << (code / 1000)) ? code % 1000 : code; }

  Vd2dArgs<T> args(const DevBuf *b, int it, int rpar, int wpar) const {
    Vd2dArgs<T> a{};
    a.nx = nx_; a.nz = nz_; a.h = h_; a.N = N_;
    a.idx = T(1.0 / c_.d.h[0]);
    a.idz = T(1.0 / c_.d.h[1]);
    a.m0 = M(0); a.m1x = M(1); a.m1z = M(2);
    a.p_o = F3(b, rpar, 0); a.vx_o = F3(b, rpar, 1); a.vz_o = F3(b, rpar, 2);
    a.p_n = F3(b, wpar, 0); a.vx_n = F3(b, wpar, 1); a.vz_n = F3(b, wpar, 2);
    a.psx_o = PSX(b, rpar); a.psx_n = PSX(b, wpar); a.spx = spx_;
    a.psz_o = PSZ(b, rpar); a.psz_n = PSZ(b, wpar); a.spz = spz_;
    a.xix_o = XIX(b, rpar); a.xix_n = XIX(b, wpar); a.sxx = sxx_;
    a.xiz_o = XIZ(b, rpar); a.xiz_n = XIZ(b, wpar); a.sxz = sxz_;
    a.cpml = cpml_.as<T>(); a.cstride = cstride_;
    a.pt = view(c_.pts);
    a.srctf = c_.pts.d_srctf.as<T>();
    a.res = c_.pts.d_res.as<T>();
    a.nt_shot = c_.pts.d_nt.as<int>();
    a.nsh = nsh_;
    a.sgrp = 1;
    a.it = it;
    a.pbuf = pbuf_.as<T>(); a.pslot = (int64_t)ns_ * N_;
    a.S = store_all_ ? (1 << 30) : S_;   // store-all: the final segment is the whole run
    const int64_t F = (int64_t)ns_ * N_;
    a.g0 = grad_.as<T>(); a.g1x = a.g0 ? a.g0 + F : nullptr; a.g1z = a.g0 ? a.g0 + 2 * F : nullptr;
    a.idt = T(1.0 / c_.d.dt);
    return a;
  }

  // 1-D grid of tiles x shots; the kernels map blocks to tiles XCD-aware
  unsigned grid(Vd2dArgs<T> &a, int tz) const {
    a.nbx = (int)ceil_div(nx_, TX);
    a.nbz = (int)ceil_div(nz_, tz);
    return (unsigned)((int64_t)a.nbx * a.nbz * nsh_);
  }

  // z-marching grid: strips of 64*W columns, chunks sized so that the
  // launch has about 2048 blocks (8 per CU) when the grid allows it
  unsigned grid_march(Vd2dArgs<T> &a, int w) const {
    a.nbx = (int)ceil_div(nx_, 64 * w);
    const int64_t per = (int64_t)a.nbx * nsh_;
    const int nbz = (int)std::max<int64_t>(1, std::min<int64_t>(ceil_div(2048, per), ceil_div(nz_, 32)));
    a.ch = (int)ceil_div(nz_, nbz);
    a.nbz = (int)ceil_div(nz_, a.ch);
    return (unsigned)((int64_t)a.nbx * a.nbz * nsh_);
  }

  // Forward variants: tile heights 8/16/32 (2-D tiles) and 102/104
  // (z-marching strips of 128/256 columns); the autotuner picks one.
  // Thousands of a 2-D tile code give the shot groups of the block order
  // (vd2d_tile_of): code + 1000 k takes groups of 2^k shots.
  void launch_fwd(Vd2dArgs<T> a, int tz) {
    a.sgrp = 1 << (used(tz) / 1000);
    tz %= 1000;
    if (tz == 102 || tz == 104) {
      const unsigned g = grid_march(a, tz - 100);
      if (tz == 102) vd2d_fwd_march<T, 2><<<g, 128, 0, c_.stream>>>(a);
      else vd2d_fwd_march<T, 4><<<g, 256, 0, c_.stream>>>(a);
      SWX_HIP(hipGetLastError());
      return;
    }
    if (tz == 208 || tz == 216 || tz == 232) {
      const unsigned g = grid(a, tz - 200);
      if (tz == 208) vd2d_fwd2_kernel<T, 8, 256><<<g, dim3(TX, 4), 0, c_.stream>>>(a);
      else if (tz == 216) vd2d_fwd2_kernel<T, 16, 512><<<g, dim3(TX, 8), 0, c_.stream>>>(a);
      else vd2d_fwd2_kernel<T, 32, 512><<<g, dim3(TX, 8), 0, c_.stream>>>(a);
      SWX_HIP(hipGetLastError());
      return;
    }
    if (tz == 408 || tz == 416) {
      // two shots per block, both kinds of tiles in one launch
      a.nbx = (int)ceil_div(nx_, TX);
      a.nbz = (int)ceil_div(nz_, tz - 400);
      const unsigned g = (unsigned)((int64_t)a.nbx * a.nbz * ceil_div(nsh_, 2));
      if (tz == 408) vd2d_fwd_pair_kernel<T, 8><<<g, dim3(TX, BY), 0, c_.stream>>>(a);
      else vd2d_fwd_pair_kernel<T, 16><<<g, dim3(TX, BY), 0, c_.stream>>>(a);
      SWX_HIP(hipGetLastError());
      return;
    }
    // 8/16/32: interior tiles, then the others (each kernel skips the other's
    // tiles); 308/316/332: one launch stepping both kinds of tiles
    const unsigned g = grid(a, tz % 100);
    const dim3 blk(TX, BY);
    switch (tz) {
      case 8: vd2d_fwd_lean<T, 8><<<g, blk, 0, c_.stream>>>(a); vd2d_fwd_kernel<T, 8, false><<<g, blk, 0, c_.stream>>>(a); break;
      case 16: vd2d_fwd_lean<T, 16><<<g, blk, 0, c_.stream>>>(a); vd2d_fwd_kernel<T, 16, false><<<g, blk, 0, c_.stream>>>(a); break;
      case 32: vd2d_fwd_lean<T, 32><<<g, blk, 0, c_.stream>>>(a); vd2d_fwd_kernel<T, 32, false><<<g, blk, 0, c_.stream>>>(a); break;
      case 308: vd2d_fwd_kernel<T, 8, true><<<g, blk, 0, c_.stream>>>(a); break;
      case 316: vd2d_fwd_kernel<T, 16, true><<<g, blk, 0, c_.stream>>>(a); break;
      default: vd2d_fwd_kernel<T, 32, true><<<g, blk, 0, c_.stream>>>(a); break;
    }
    SWX_HIP(hipGetLastError());
  }
  // Windows of vd2d_stepn_kernel: rows per wave and waves per block of shape 0
  // (forward, few windows), 1 (forward, many) and 2 (adjoint), all 64 columns
  // wide; as high as registers allow for the number of waves.
  struct Shape {
    int r, nw;
  };
  static constexpr Shape SHAPES[3] = {{4, sizeof(T) == 4 ? 16 : 8}, {6, sizeof(T) == 4 ? 16 : 8},
                                      {sizeof(T) == 4 ? 8 : 4, 8}};
  static constexpr int NMAX = std::min(SN_MAX, (SHAPES[0].r * SHAPES[0].nw - 1) / 6);   // most levels of a window
  int64_t stepn_blocks(int shape, int n) const {
    return std::max<int64_t>(ceil_div(nx_ - 6 * n, TX - 6 * n), 1) *
           std::max<int64_t>(ceil_div(nz_ - 6 * n, SHAPES[shape].r * SHAPES[shape].nw - 6 * n), 1) * nsh_;
  }
  template <int S, bool ADJ>
  void launch_shape(Vd2dArgs<T> a, int n) {
    constexpr int R = SHAPES[S].r, NW = SHAPES[S].nw;
    a.nbx = (int)std::max<int64_t>(ceil_div(nx_ - 6 * n, TX - 6 * n), 1);
    a.nbz = (int)std::max<int64_t>(ceil_div(nz_ - 6 * n, R * NW - 6 * n), 1);
    vd2d_stepn_kernel<T, R, NW, ADJ><<<(unsigned)stepn_blocks(S, n), TX * NW, 0, c_.stream>>>(a, n);
    SWX_HIP(hipGetLastError());
  }
  void launch_stepn(const Vd2dArgs<T> &a, int n, bool adj) {
    if (adj) launch_shape<2, true>(a, n);
    else if (tz_fwd_ > 510) launch_shape<1, false>(a, n);
    else launch_shape<0, false>(a, n);
  }
  void launch_adj(Vd2dArgs<T> a, int tz) {
    a.sgrp = 1 << (used(tz) / 1000);
    tz %= 1000;
    if (tz == 102 || tz == 104) {
      const unsigned g = grid_march(a, tz - 100);
      if (tz == 102) vd2d_adj_march<T, 2><<<g, 128, 0, c_.stream>>>(a);
      else vd2d_adj_march<T, 4><<<g, 256, 0, c_.stream>>>(a);
      SWX_HIP(hipGetLastError());
      return;
    }
    if (tz == 416) {
      // two shots per block, both kinds of tiles in one launch
      a.nbx = (int)ceil_div(nx_, TX);
      a.nbz = (int)ceil_div(nz_, 16);
      const unsigned g = (unsigned)((int64_t)a.nbx * a.nbz * ceil_div(nsh_, 2));
      vd2d_adj_pair_kernel<T, 16><<<g, dim3(TX, BY), 0, c_.stream>>>(a);
      SWX_HIP(hipGetLastError());
      return;
    }
    // 8/16: interior tiles, then the others; 308/316: one launch
    const unsigned g = grid(a, tz % 100);
    const dim3 blk(TX, BY);
    switch (tz) {
      case 8: vd2d_adj_lean<T, 8><<<g, blk, 0, c_.stream>>>(a); vd2d_adj_kernel<T, 8, false><<<g, blk, 0, c_.stream>>>(a); break;
      case 16: vd2d_adj_lean<T, 16><<<g, blk, 0, c_.stream>>>(a); vd2d_adj_kernel<T, 16, false><<<g, blk, 0, c_.stream>>>(a); break;
      case 308: vd2d_adj_kernel<T, 8, true><<<g, blk, 0, c_.stream>>>(a); break;
      default: vd2d_adj_kernel<T, 16, true><<<g, blk, 0, c_.stream>>>(a); break;
    }
    SWX_HIP(hipGetLastError());
    SWX_HIP(hipGetLastError());
  }

  Vd2dArgs<T> fwd_args(int it, int act_min, int smode, int cbase, T *traces) const {
    Vd2dArgs<T> a = args(st_, it, slot(it - 1), slot(it));
    a.act_min = act_min;
    a.smode = smode;
    a.cbase = cbase;
    a.traces = traces;
    return a;
  }
  Vd2dArgs<T> adj_args(int it, int cbase) const {
    Vd2dArgs<T> a = args(ad_, it, (it + 1 + aflip_) & 1, (it + aflip_) & 1);
    a.cbase = cbase;
    return a;
  }

  // steps it .. it+n-1 in one launch
  void fwd_step(int it, int n, int act_min, int smode, int cbase, T *traces) {
    const Vd2dArgs<T> a = fwd_args(it, act_min, smode, cbase, traces);
    c_.ktimer.begin(c_.stream);
    if (is_stepn(tz_fwd_)) {
      launch_stepn(a, n, false);
    } else {
      // the last step before a checkpoint (or of a replay) runs the
      // single-step kernel of the same tile height
      launch_fwd(a, steps_per_launch(tz_fwd_) == 2 && n == 1 ? tz_fwd_ - 200 : tz_fwd_);
    }
    if (n % 2 == 0) flip_ ^= 1;
    c_.ktimer.end(c_.stream, 0);
  }

  // adjoint steps it .. it-n+1 in one launch
  void adj_step(int it, int n, int cbase) {
    const Vd2dArgs<T> a = adj_args(it, cbase);
    c_.ktimer.begin(c_.stream);
    if (is_stepn(tz_adj_)) launch_stepn(a, n, true);
    else launch_adj(a, tz_adj_);
    if (n % 2 == 0) aflip_ ^= 1;
    c_.ktimer.end(c_.stream, 1);
  }

  // Levels per launch (code 500 + levels; 510 + levels: shape 1), or 0: one,
  // with a tuned tile.  A launch of few windows costs a level's latency whatever
  // their number, up to one block per CU, so that the most levels whose windows
  // still number at most 256 are the best.  Beyond, the halos count: the forward
  // takes the taller windows of shape 1, and 4 levels (float32) or 3 (float64,
  // half the rows) balance them against the launches; the adjoint, which its
  // registers hold to the height of shape 0, takes 3, and in float64 2 and at
  // last single steps.  us per level, forward: best tile / 3 / 4 / 5 / 6 levels /
  // shape 1 with 3 / 4 / 5:
  //   f32  300 x 200, 4 shots     9.9 / 5.2 / 4.5 / 3.9 / 3.7 / 6.1 / 5.2 / 4.5
  //   f32  701 x 403              9.7 / 5.1 / 4.4 / 3.8 /   - / 6.1 / 5.1 / 4.5
  //   f32  1000 x 1000           14.6 / 8.5 / 9.8 /  11 /   - /  10 / 8.6 / 8.0
  //   f32  800 x 600, 3 shots    18.1 /  12 /  13 /   - /   - /  11 / 9.9 /  11
  //   f32  1000 x 700, 8 shots     49 /  38 /  41 /  49 /   - /  33 /  33 /  36
  //   f32  2000 x 800, 32 shots   349 / 315 / 344 / 401 / 530 / 296 / 270 / 291
  //   f64  331 x 257              9.6 / 5.4 / 4.5 /  12 /   - / 5.9 / 5.1 / 4.5
  //   f64  331 x 257, 8 shots    17.4 /  15 /  21 /  70 /   - /  11 /  12 /  14
  //   f64  1000 x 1000           20.8 /  20 /  30 / 110 /   - /  15 /  17 /  21
  //   f64  1000 x 700, 8 shots     86 /  97 / 151 /   - /   - /  71 /  78 / 102
  // Adjoint with replay (forward as chosen above): tile / 2 / 3 / 4 levels
  //   f32  701 x 403             15.8 /  14 /  11 / 9.8   (5: 9.0)
  //   f32  2000 x 800, 32 shots   864 / 830 / 751 / 746
  //   f64  331 x 257             17.2 /  12 /  10 / 9.1
  //   f64  1000 x 1000             47 /  38 /  41 /  53
  //   f64  1000 x 700, 8 shots    202 / 201 / 207 / 273
  // Next to the two lines (910 and 1078 windows of 3 levels, 2660 and 3990 of 2;
  // the second line lies a little before the last gain of two levels):
  //   f64  600 x 500, 2 shots    35.2 / 27.5 / 27.3
  //   f64  1000 x 700            36.5 / 30.0 / 31.5
  //   f64  1000 x 700, 4 shots    110 / 105 / 107
  //   f64  1000 x 700, 6 shots    158 / 154 / 156
  int choose_steps(const char *env, bool adj) const {
    if (const char *v = std::getenv(env)) {
      const int t = std::atoi(v);
      return (t / 10 == 50 || (t / 10 == 51 && !adj)) && t % 10 >= 1 && t % 10 <= NMAX ? t : 0;
    }
    const bool f32 = sizeof(T) == 4;
    for (int n = f32 ? 6 : 4; n > 3; n--)
      if (stepn_blocks(0, n) <= 256) return 500 + n;
    if (!adj) return f32 ? 514 : 513;
    if (f32 || stepn_blocks(2, 3) <= 1024) return 503;
    return stepn_blocks(2, 2) <= 3072 ? 502 : 0;
  }

  // Tuner candidates: the 2-D tile heights 8/16/32 as an interior-tile launch
  // plus an other-tile launch, the same heights as one launch (308/316/332),
  // and the z-marching strips (codes 102/104) when kMarchInTuner is set.
  // The adjoint times tile height 16 only: on the 64-shot batch the height-8
  // variants measured 15% slower over whole runs, but the short tuning
  // window could not tell them apart reliably.  The environment can
  // pin any variant, including two steps per launch (208/216/232 for tile
  // heights 8/16/32), which measured slower per step than one step per
  // launch on MI355X and is therefore not timed by default.
  static constexpr bool kMarchInTuner = false;
  static std::vector<int> candidates(std::vector<int> tiles) {
    if (kMarchInTuner) {
      tiles.push_back(102);
      tiles.push_back(104);
    }
    return tiles;
  }

  // Times each candidate tile height on a real launch (a step depends only
  // on the previous parity, so repeating it is harmless; the adjoint tuning
  // runs before the adjoint state and gradients are cleared) and returns the
  // fastest.  The candidates are timed in three interleaved rounds of five
  // launches and each keeps its best round, so a clock ramp or a busy
  // moment during one round does not decide.  The shot groups of the block
  // order (code + 1000 k) are then timed for the fastest 2-D tile variant.
  // SWX_VD2D_TILE_FWD / _ADJ pin a value instead (also the variants the
  // tuner does not time: the
  // z-marching strips 102/104, two steps per launch 208/216/232 and two
  // shots per block 408/416, all measured slower on MI355X).
  template <typename F>
  int tune(const char *env, const std::vector<int> &cands, F launch) {
    if (const char *v = std::getenv(env)) {
      const int t = std::atoi(v), base = t % 1000, k = t / 1000;
      for (int c : cands)
        if (c == base && (k == 0 || (k <= 3 && nsh_ % (1 << k) == 0))) return t;
      if (t == 102 || t == 104 || t == 208 || t == 216 || t == 232 || t == 408 || t == 416) return t;
    }
    // the tile variant in the plain shot order, then its shot groups
    const int tile = fastest(cands, launch);
    return fastest(with_groups(tile), launch);
  }
  template <typename F>
  int fastest(const std::vector<int> &cands, F launch) {
    if (cands.size() == 1) return cands.front();
    progress("launch shapes timed", 1, 1);
    hipEvent_t e0, e1;
    SWX_HIP(hipEventCreate(&e0));
    SWX_HIP(hipEventCreate(&e1));
    std::vector<float> best_of(cands.size(), 1e30f);
    for (size_t c = 0; c < cands.size(); c++) launch(cands[c]);
    for (int round = 0; round < 3; round++) {
      for (size_t c = 0; c < cands.size(); c++) {
        SWX_HIP(hipEventRecord(e0, c_.stream));
        for (int r = 0; r < 5; r++) launch(cands[c]);
        SWX_HIP(hipEventRecord(e1, c_.stream));
        SWX_HIP(hipEventSynchronize(e1));
        float ms = 0;
        SWX_HIP(hipEventElapsedTime(&ms, e0, e1));
        ms /= (float)steps_per_launch(cands[c]);   // per time step
        best_of[c] = std::min(best_of[c], ms);
      }
    }
    int best = cands.front();
    float bestms = 1e30f;
    for (size_t c = 0; c < cands.size(); c++)
      if (best_of[c] < bestms) { bestms = best_of[c]; best = cands[c]; }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    return best;
  }
  int tz_fwd_ = 0, tz_adj_ = 0;          // codes of the batch in hand
  int tile_fwd_ = 0, tile_adj_ = 0;      // timed once per plan, kept through batches that take several levels
  int flip_ = 0, aflip_ = 0;

  // checkpoint k (k = 1 .. floor(nt_max/S), all shots): p, vx, vz, psi_x,
  // psi_z, xi_x, xi_z at parity cb&1
  void ckpt_copy(int k, int cb, bool save) {
    const int64_t e = sizeof(T);
    const int par = slot(cb);
    char *base = ck_.as<char>() + (int64_t)(k - 1) * ck_one_;
    struct Part { void *dev; int64_t bytes; };
    const Part parts[5] = {
        {F3(st_, par, 0), 3 * ns_ * N_ * e},
        {PSX(st_, par), ns_ * spx_ * e},
        {PSZ(st_, par), ns_ * spz_ * e},
        {XIX(st_, par), ns_ * sxx_ * e},
        {XIZ(st_, par), ns_ * sxz_ * e},
    };
    int64_t off = 0;
    for (const Part &pt : parts) {
      if (pt.bytes) {
        if (save) SWX_HIP(hipMemcpyAsync(base + off, pt.dev, pt.bytes, hipMemcpyDeviceToDevice, c_.stream));
        else SWX_HIP(hipMemcpyAsync(pt.dev, base + off, pt.bytes, hipMemcpyDeviceToDevice, c_.stream));
      }
      off += pt.bytes;
    }
  }

  PlanCore &c_;
  int nx_, nz_, h_, ns_;
  int64_t N_, spx_, spz_, sxx_, sxz_;
  int cstride_;
  DevBuf m_, cpml_;
  DevBuf st_[3], ad_[3];   // [0] p/vx/vz, [1] psi, [2] xi; both parities
  DevBuf grad_, gout_, pbuf_, ck_;
  int64_t ck_one_ = 0, state_bytes_ = 0;
  int S_ = 1, K_ = 1, nck_ = 0;
  bool store_all_ = true;
  int nsh_ = 0, ntmax_ = 0;
  std::vector<int> nt_;
  bool model_set_ = false;
};

}  // namespace

std::unique_ptr<Engine> make_acoustic_vd2d(PlanCore &core) {
  if (core.d.dtype == SWX_F32) return std::make_unique<Vd2dEngine<float>>(core);
  return std::make_unique<Vd2dEngine<double>>(core);
}

}  // namespace swx
