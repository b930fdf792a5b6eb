// 2D acoustic constant-density engine: fused C-PML time step, point
// (source/receiver) kernel, checkpoint/replay driver and gradient
// correlation for a batch of shots.
//
// Reference semantics (paths relative to the reference root):
//   step       src/models/acoustic/backends/shared/acoustic2D_xPU.jl:1-169
//   stencils   src/utils/fdgen.jl:137-193 (order 2)
//   driver     src/models/acoustic/acou_gradient.jl:4-95
//   correlate  src/models/acoustic/backends/shared/correlate_gradient_xPU.jl:1-10
//
// Device layout (x fastest, exactly the Julia layout), one slab per shot:
//   p      [4][ns][nx*nz]  the two last time levels and the slots of the
//                          next two (the reference swaps pold/pcur/pnew,
//                          :122-124)
//   psi_x  [3][ns][2h*nz]  the last level and free buffers for the next, so a
//   psi_z  [3][ns][nx*2h]  cell can recompute its left neighbour's new value
//   xi_x   [3][ns][(2h+2)*nz], xi_z [3][ns][nx*(2h+2)]
//   (the adjoint state is laid out the same way)
//   D      [S][ns][nx*nz]  p^{it-2} - 2 p^{it-1} + p^{it} of the segment
//                          being replayed (what correlate_gradient! needs)
//   ckpt   [K-2][...]      p^{c-1}, p^c, psi, xi at c = k*S
//   grad   [ns][nx*nz]     per-shot raw gradient (reduced in shot order)
#include <algorithm>
#include <cstdlib>
#include <mutex>

#include <hip/hip_ext.h>

#include "swx_levels.hpp"
#include "swx_internal.hpp"

namespace swx {
namespace {

constexpr int TX = 64;  // one wavefront along the fast axis
constexpr int TZ = 4;   // waves per block; each thread steps R rows TZ apart

template <typename T>
struct Cd2dStepArgs {
  int nx, nz, h;
  int64_t N;                 // nx*nz
  T idx, idz, idx2, idz2;
  const T *__restrict__ fact;
  const T *pold;             // shot 0 slab of the three time levels
  const T *pcur;
  T *pnew;
  const T *psix_o; T *psix_n; int64_t spx;   // psi_x old/new, per-shot stride
  const T *psiz_o; T *psiz_n; int64_t spz;
  const T *xix_o; T *xix; int64_t sxx;   // xi_x of the previous / this level (may be one array)
  const T *xiz_o; T *xiz; int64_t sxz;
  const T *cpml; int cstride;                // per-shot packed coefficients
  const int *nt_shot;
  int it;                    // time step index (1-based)
  int act_min;               // shot active iff it <= nt_s and nt_s > act_min
  // D store: dmode 0 none, 1 forward last segment, 2 replay slot it-cbase-1
  T *dbuf; int64_t dslot; int dmode; int S; int cbase;
  // correlation of the current (adjoint) field with D slot it-cbase
  T *grad; int corr; int corr_lim;
  // sources/receivers: forward injects srctf and records traces (nullable);
  // the adjoint (res != nullptr) injects the residuals prescaled by fact
  PointArgsView pt;
  const T *srctf;
  T *traces;
  const T *res;
  int nbx, nby;              // tiles of TX x (TZ * R) cells along x, z
  int lean;                  // interior tiles take cd2d_lean_cells
};

// Block -> tile map giving each of the 8 XCDs a contiguous run of tiles, so
// the halo lines neighbouring tiles share are found in one L2.
__device__ __forceinline__ int xcd_tile2(int b, int nb) {
  const int per = nb >> 3;
  if (b >= per * 8) return b;
  return (b & 7) * per + (b >> 3);
}

// Interior tile: every cell of rows J0..J1 and columns I0..I0+TX-1 takes the
// plain Laplacian branch (inside the grid, outside the C-PML strips, no
// memory variable owned) and no point of the launch's families lies on
// those rows.
template <typename T>
__device__ __forceinline__ bool cd2d_is_lean(const Cd2dStepArgs<T> &a, int s, int I0, int J0, int J1) {
  const int nx = a.nx, nz = a.nz, h = a.h;
  if (!(I0 >= max(h, 1) && I0 + TX - 1 <= nx - h - 2 && J0 >= max(h, 1) && J1 <= nz - h - 2)) return false;
  const int64_t o = (int64_t)s * (a.pt.nrows + 1);
  const int *rowp = a.res == nullptr ? a.pt.srow : a.pt.rrow;
  if (rowp[o + J0] != rowp[o + J1 + 1]) return false;
  if (a.traces && a.pt.rrow[o + J0] != a.pt.rrow[o + J1 + 1]) return false;
  return true;
}

// R cells (i, J0 + r * TZ) of an interior tile: every load of the R cells is
// issued before the first store; the expressions are those of cd2d_cell's
// interior branch, so results are bitwise equal.
template <typename T, int R>
__device__ __forceinline__ void cd2d_lean_cells(const Cd2dStepArgs<T> &a, int s, int nts, int i, int J0) {
  const int nx = a.nx;
  const int64_t so = (int64_t)s * a.N;
  const T *__restrict__ pc_ = a.pcur + so;
  const T *__restrict__ po_ = a.pold + so;
  T *__restrict__ pn_ = a.pnew + so;
  const bool corr = a.corr && a.it + 1 <= nts && a.it + 1 <= a.corr_lim;
  int slot = -1;
  if (a.dmode == 1) {
    const int seg0 = ((nts - 1) / a.S) * a.S;
    if (a.it > seg0) slot = a.it - seg0 - 1;
  } else if (a.dmode == 2) {
    slot = a.it - a.cbase - 1;
  }
  const T *dsrc = corr ? a.dbuf + (int64_t)(a.it - a.cbase) * a.dslot + so : nullptr;
  T pc[R], pl[R], pr[R], pd[R], pu[R], pov[R], fa[R], gv[R], dv[R];
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int c = (J0 + r * TZ) * nx + i;
    pc[r] = pc_[c];
    pl[r] = pc_[c - 1];
    pr[r] = pc_[c + 1];
    pd[r] = pc_[c - nx];
    pu[r] = pc_[c + nx];
    pov[r] = po_[c];
    fa[r] = a.fact[c];
    gv[r] = corr ? a.grad[so + c] : T(0);
    dv[r] = corr ? dsrc[c] : T(0);
  }
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int c = (J0 + r * TZ) * nx + i;
    const T d2x = (pl[r] - T(2) * pc[r] + pr[r]) * a.idx2;
    const T d2z = (pd[r] - T(2) * pc[r] + pu[r]) * a.idz2;
    const T lx = d2x, lz = d2z;
    const T flap = fa[r] * (lx + lz);
    const T pnv = T(2) * pc[r] - pov[r] + flap;
    const T inj = 0;
    pn_[c] = pnv;
    if (slot >= 0) a.dbuf[(int64_t)slot * a.dslot + so + c] = flap + inj;
    if (corr) a.grad[so + c] = gv[r] + pc[r] * dv[r];
  }
}

// One cell of the step: C-PML memory variables, Laplacian, points, replay
// history and correlation.
template <typename T>
__device__ __forceinline__ void cd2d_cell(const Cd2dStepArgs<T> &a, int s, int nts, int i, int j) {
  const int nx = a.nx, nz = a.nz, h = a.h;
  if (i >= nx || j >= nz) return;
  const int64_t so = (int64_t)s * a.N;
  const int64_t c = (int64_t)j * nx + i;
  const T *pc_ = a.pcur + so;
  const T *po_ = a.pold + so;
  T *pn_ = a.pnew + so;
  const bool interior = (i >= 1 && i <= nx - 2 && j >= 1 && j <= nz - 2);
  const bool corr = a.corr && a.it + 1 <= nts && a.it + 1 <= a.corr_lim;
  // the loads that do not depend on a branch's outcome are issued together
  const T pc = pc_[c];
  const T pl = interior ? pc_[c - 1] : T(0), pr = interior ? pc_[c + 1] : T(0);
  const T pd = interior ? pc_[c - nx] : T(0), pu = interior ? pc_[c + nx] : T(0);
  const T pov = po_[c], fa = a.fact[c];
  const T gv = corr ? a.grad[so + c] : T(0);
  const T dv = corr ? a.dbuf[(int64_t)(a.it - a.cbase) * a.dslot + so + c] : T(0);
  const T *cb = a.cpml + (int64_t)s * a.cstride;
  const AxisCoef<T> cx = axis_coef(cb, h, 0);
  const AxisCoef<T> cz = axis_coef(cb, h, 1);

  // psi_x: cell i owns strip index kx (update_psi_x!, acoustic2D_xPU.jl:1-12)
  int kx = -1;
  if (i < h) kx = i;
  else if (i >= nx - h - 1 && i <= nx - 2) kx = i + 1 - nx + 2 * h;
  T psx = 0;
  if (kx >= 0) {
    const int64_t q = (int64_t)s * a.spx + (int64_t)j * (2 * h) + kx;
    const T d = (pc_[c + 1] - pc) * a.idx;
    psx = cx.bh(kx) * a.psix_o[q] + cx.ah(kx) * d;
    a.psix_n[q] = psx;
  }
  // psi_z (update_psi_y!, acoustic2D_xPU.jl:14-25)
  int kz = -1;
  if (j < h) kz = j;
  else if (j >= nz - h - 1 && j <= nz - 2) kz = j + 1 - nz + 2 * h;
  T psz = 0;
  if (kz >= 0) {
    const int64_t q = (int64_t)s * a.spz + (int64_t)kz * nx + i;
    const T d = (pc_[c + nx] - pc) * a.idz;
    psz = cz.bh(kz) * a.psiz_o[q] + cz.ah(kz) * d;
    a.psiz_n[q] = psz;
  }

  T pnv = 0, flap = 0, inj = 0;
  if (interior) {
    // update_p_CPML! (acoustic2D_xPU.jl:27-46)
    const T d2x = (pl - T(2) * pc + pr) * a.idx2;
    const T d2z = (pd - T(2) * pc + pu) * a.idz2;
    T lx = d2x, lz = d2z;
    if (i < h || i >= nx - h) {
      // left neighbour's new psi, recomputed from the old buffer
      const int kn = kx - 1;
      const int64_t qn = (int64_t)s * a.spx + (int64_t)j * (2 * h) + kn;
      const T psn = cx.bh(kn) * a.psix_o[qn] + cx.ah(kn) * ((pc - pl) * a.idx);
      const T dpsi = (psx - psn) * a.idx;
      const int64_t qx = (int64_t)s * a.sxx + (int64_t)j * (2 * h + 2) + kx;
      const T xi = cx.b(kx) * a.xix_o[qx] + cx.a(kx) * (d2x + dpsi);
      a.xix[qx] = xi;
      lx = d2x + dpsi + xi;
    }
    if (j < h || j >= nz - h) {
      const int kn = kz - 1;
      const int64_t qn = (int64_t)s * a.spz + (int64_t)kn * nx + i;
      const T psn = cz.bh(kn) * a.psiz_o[qn] + cz.ah(kn) * ((pc - pd) * a.idz);
      const T dpsi = (psz - psn) * a.idz;
      const int64_t qz = (int64_t)s * a.sxz + (int64_t)kz * nx + i;
      const T xi = cz.b(kz) * a.xiz_o[qz] + cz.a(kz) * (d2z + dpsi);
      a.xiz[qz] = xi;
      lz = d2z + dpsi + xi;
    }
    flap = fa * (lx + lz);
    pnv = T(2) * pc - pov + flap;
  }
  // Edge cells are outside the stencil range.  The reference's rotation
  // (acoustic2D_xPU.jl:122-124) binds pnew to the array of the new pold, so
  // an edge cell of level it holds level it-2 plus what is injected there.
  if (!interior) pnv = pov;
  // Points of this cell: inject_sources! / record_receivers! (forward,
  // acoustic2D_xPU.jl:48-62) or the prescaled residual injection of the
  // adjoint (:64-76, :161-162), in the reference's serial order per cell.
  if (a.res == nullptr) {
    const int u = find_point(a.pt.srow, a.pt.usrc_cell, a.pt.nrows, s, j, c);
    if (u >= 0) {
      const T *tf = a.srctf + a.pt.off_tf[s] + (a.it - 1);
      for (int k = a.pt.usrc_ptr[u]; k < a.pt.usrc_ptr[u + 1]; k++) {
        const T v = tf[(int64_t)nts * a.pt.usrc_list[k]];
        pnv += v;
        inj += v;
      }
    }
  } else {
    const int u = find_point(a.pt.rrow, a.pt.urec_cell, a.pt.nrows, s, j, c);
    if (u >= 0) {
      const T *rs = a.res + a.pt.off_tr[s] + (a.it - 1);
      const T f = fa;
      for (int k = a.pt.urec_ptr[u]; k < a.pt.urec_ptr[u + 1]; k++) pnv += rs[(int64_t)nts * a.pt.urec_list[k]] * f;
    }
  }
  pn_[c] = pnv;
  if (a.traces) {
    const int r = find_point(a.pt.rrow, a.pt.urec_cell, a.pt.nrows, s, j, c);
    if (r >= 0) {
      T *tr = a.traces + a.pt.off_tr[s] + (a.it - 1);
      for (int k = a.pt.urec_ptr[r]; k < a.pt.urec_ptr[r + 1]; k++) tr[(int64_t)nts * a.pt.urec_list[k]] = pnv;
    }
  }
  if (a.dmode) {
    int slot = -1;
    if (a.dmode == 1) {
      const int seg0 = ((nts - 1) / a.S) * a.S;
      if (a.it > seg0) slot = a.it - seg0 - 1;
    } else {
      slot = a.it - a.cbase - 1;
    }
    if (slot >= 0) {
      // p^{it} - 2 p^{it-1} + p^{it-2}: in the interior exactly the stencil
      // term plus the injection, formed without cancellation
      a.dbuf[(int64_t)slot * a.dslot + so + c] = interior ? flap + inj : (pov - T(2) * pc) + pnv;
    }
  }
  if (corr) {
    // correlate_gradient! of the previous adjoint step (adjcur = pcur here)
    a.grad[so + c] = gv + pc * dv;
  }
}

// One time step on a tile of TX x (TZ * R) cells per block (a 1D grid of
// nbx * nby * shots blocks, dealt to the XCDs in contiguous runs).
template <typename T, int R>
__global__ __launch_bounds__(TX *TZ) void cd2d_step_kernel(Cd2dStepArgs<T> a) {
  const int b = xcd_tile2(blockIdx.x, gridDim.x);
  const int t = b / a.nbx;
  const int bx = b - t * a.nbx, by = t % a.nby, s = t / a.nby;
  const int nts = a.nt_shot[s];
  if (a.it > nts || nts <= a.act_min) return;
  const int i = bx * TX + threadIdx.x;
  const int J0 = by * TZ * R;
  if (a.lean && cd2d_is_lean(a, s, bx * TX, J0, J0 + TZ * R - 1)) {
    cd2d_lean_cells<T, R>(a, s, nts, i, J0 + threadIdx.y);
    return;
  }
  for (int r = 0; r < R; r++) cd2d_cell(a, s, nts, i, J0 + threadIdx.y + r * TZ);
}

// ---------------------------------------------------------------------------
// Up to SN_MAX levels per launch (cd2d_stepn_kernel).
//
// A block of NW waves loads a 64 x (NW R) window of the two last levels
// into registers (lane = column, R rows per wave) and steps it n times; the
// window's valid part shrinks by one cell per level and side, so the block
// owns, and writes, the cells at least n from the window's sides (all cells
// up to a side that is the grid's).  x neighbours come from the adjacent
// lanes, z neighbours from the thread's own rows; only the first and last row
// of each wave pass through LDS, with one barrier per level.  The C-PML
// memory variables of the window's strip cells step along in registers, and
// in the adjoint the gradient of the owned cells, with the forward history
// loaded two levels ahead.  Point values of the n levels are staged in LDS
// once.  Every cell update is spelled as in cd2d_cell, so the results are
// bitwise those of n one-level launches.
//
// Bound by latency: of the barrier, the LDS round trip and the strip updates'
// chain of a level, and of a launch's loads and stores (one 201 x 151 shot:
// 11.3 us per launch of 8 levels).  Counters, forward / adjoint: 1000 x 1000
// float32 has 1.2 / 1.8 waves per SIMD, vector units issuing 0.22 of the time,
// 1.5 / 2.5 TB/s; 4 x 2000 x 1000 has 3.0 / 3.2, 0.48 / 0.38 and 2.7 / 3.6 TB/s,
// with 1.5-1.8 times the grid's cells stepped.  us per level against the
// two-level LDS tiles this replaces (one level per launch where that was
// faster):
//   f32 201 x 151:        forward 5.1 -> 1.8, adjoint + replay   8.9 -> 3.2
//   f32 1000 x 1000:      forward 7.9 -> 3.5, adjoint + replay  15.9 -> 7.6
//   f64 12 x 397 x 253:   forward  15 -> 6.0, adjoint + replay    33 -> 15

template <typename T>
struct Cd2dStepNArgs {
  Cd2dStepArgs<T> a;   // a.it: first level; a.pnew: the last level stepped
  T *pnew0;            // the level before it (n >= 2)
  int n;               // levels
};

template <typename T, int R, int NW>
struct Cd2dNLds : LevelPoints<T, NW * R> {
  T first[2][NW][TX], last[2][NW][TX], lastz[2][NW][TX];   // rows 0 and R-1 of p, row R-1 of psi_z
  T cz[NW * R + 1][4];         // z C-PML coefficients b_h, a_h, b, a of the rows, from the one before
};

// Registers of one thread: R cells of a column.
template <typename T, int R>
struct Cd2dNRegs {
  T pc[R], po[R], fa[R];
  T psx[R], xix[R], psz[R], xiz[R];
};

// One level on a thread's R cells.  XS: the window reaches an x strip or x
// edge; ZS: the wave's rows reach a z strip or z edge.  up / dn: values of
// the row before the first / after the last, zup: old psi_z of the row
// before.  dv receives what the history keeps of a forward level (before the
// injection).
template <typename T, int R, int NW, bool ADJ, bool XS, bool ZS>
__device__ __forceinline__ void cd2d_n_level(const Cd2dStepArgs<T> &a, const Cd2dNLds<T, R, NW> &L,
                                             const LevelWin &W, int kx, const T *xc, T up, T dn, T zup,
                                             Cd2dNRegs<T, R> &G, T *dv) {
  const int nx = a.nx, h = a.h, i = W.i;
  const bool xin = !XS || (i >= 1 && i <= nx - 2);
  const bool xst = XS && (i < h || i >= nx - h);
  T prev = up, pszp = 0;
#pragma unroll
  for (int r = 0; r < R; r++) {
    const bool interior = xin && (!ZS || (W.jin >> r & 1));
    const T pc = G.pc[r], pov = G.po[r];
    const T pl = lane_before(pc), pr = lane_after(pc);
    const T pd = prev, pu = r + 1 < R ? G.pc[r + 1 < R ? r + 1 : r] : dn;
    const T d2x = (pl - T(2) * pc + pr) * a.idx2;
    const T d2z = (pd - T(2) * pc + pu) * a.idz2;
    T lx = d2x, lz = d2z;
    if (XS) {
      // psi_x of the cell's own strip entry; the left neighbour's is its lane's
      const T d = (pr - pc) * a.idx;
      const T psx = kx >= 0 ? xc[0] * G.psx[r] + xc[1] * d : T(0);
      const T psn = lane_before(psx);
      G.psx[r] = psx;
      if (xst && interior) {
        const T dpsi = (psx - psn) * a.idx;
        const T xi = xc[2] * G.xix[r] + xc[3] * (d2x + dpsi);
        G.xix[r] = xi;
        lx = d2x + dpsi + xi;
      }
    }
    if (ZS) {
      T psz = 0;
      if (W.kzr >> r & 1) {
        const T *cz = L.cz[W.w * R + r + 1];
        const T d = (pu - pc) * a.idz;
        psz = cz[0] * G.psz[r] + cz[1] * d;
        if (W.xzr >> r & 1) {
          // psi_z of the row before: stepped already, or (first row of the
          // wave) recomputed from its old value
          T psn = pszp;
          if (r == 0) {
            const T dp = (pc - pd) * a.idz;
            psn = cz[-4] * zup + cz[-3] * dp;
          }
          if (interior) {
            const T dpsi = (psz - psn) * a.idz;
            const T xi = cz[2] * G.xiz[r] + cz[3] * (d2z + dpsi);
            G.xiz[r] = xi;
            lz = d2z + dpsi + xi;
          }
        }
      }
      G.psz[r] = psz;
      pszp = psz;
    }
    const T flap = G.fa[r] * (lx + lz);
    T pnv = T(2) * pc - pov + flap;
    T dval = flap;
    if (XS || ZS) {
      if (!interior) {
        pnv = pov;
        dval = (pov - T(2) * pc) + pnv;
      }
    }
    prev = pc;
    G.po[r] = pc;
    G.pc[r] = pnv;
    if (!ADJ) dv[r] = dval;
  }
}

// Forward / replay levels it .. it+n-1, or (ADJ) adjoint levels it .. it-n+1
// with their injection and their correlation with the forward history.
template <typename T, int R, int NW, bool ADJ>
__global__ __launch_bounds__(NW *TX, sizeof(T) == 4 ? 4 : 2) void cd2d_stepn_kernel(Cd2dStepNArgs<T> A) {
  const Cd2dStepArgs<T> &a = A.a;
  __shared__ Cd2dNLds<T, R, NW> L;
  constexpr int H = NW * R;
  if (threadIdx.x == 0) L.used = L.rused = 0;
  __syncthreads();
  const int b = xcd_tile2(blockIdx.x, gridDim.x);
  const int t = b / a.nbx;
  const int bx = b - t * a.nbx, by = t % a.nby, s = t / a.nby;
  const int nts = a.nt_shot[s];
  const int n = A.n, nx = a.nx, nz = a.nz, h = a.h;
  const int X0 = bx * (TX - 2 * n), Z0 = by * (H - 2 * n);
  LevelWin W;
  W.lane = threadIdx.x & (TX - 1);
  W.w = __builtin_amdgcn_readfirstlane(threadIdx.x / TX);
  W.i = X0 + W.lane;
  W.j0 = Z0 + W.w * R;
  W.own = W.i < nx && W.lane >= (bx ? n : 0) && W.lane < (bx < a.nbx - 1 ? TX - n : TX);
  W.rows = W.jin = W.kzr = W.xzr = 0;
  const int own0 = by ? Z0 + n : 0, own1 = by < a.nby - 1 ? Z0 + H - n : nz;
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int j = W.j0 + r;
    if (j >= own0 && j < own1) W.rows |= 1 << r;
    if (j >= 1 && j <= nz - 2) {
      W.jin |= 1 << r;
      if (j < h || j >= nz - h) W.xzr |= 1 << r;
    }
    if (j < h || (j >= nz - h - 1 && j <= nz - 2)) W.kzr |= 1 << r;
  }
  const int64_t so = (int64_t)s * a.N;
  const bool xs = X0 < max(h, 1) || X0 + TX - 1 >= nx - h - 1;
  const bool zs = W.j0 < max(h, 1) || W.j0 + R - 1 >= nz - h - 1;
  int kx = -1;
  if (W.i < h) kx = W.i;
  else if (W.i >= nx - h - 1 && W.i <= nx - 2) kx = W.i + 1 - nx + 2 * h;

  Cd2dNRegs<T, R> G;
  T g[R], d0[R], d1[R];
  const T *pc_ = a.pcur + so, *po_ = a.pold + so;
  // Rows and columns beyond the grid take those of its edge: what they hold
  // is never read by a cell of the grid (edge cells read no neighbour).
  const unsigned ic = min(W.i, nx - 1);
  auto row = [&](const T *p, int r) { return p + (int64_t)min(W.j0 + r, nz - 1) * nx; };
  auto strip = [&](int r) {      // z strip entry of row r
    const int j = W.j0 + r;
    return j < h ? j : j + 1 - nz + 2 * h;
  };
  // forward history of level l (ADJ)
  auto fetch = [&](T *d, int l) {
    const T *slot = a.dbuf + (int64_t)(max(l, a.it - n + 1) - a.cbase - 1) * a.dslot + so;
#pragma unroll
    for (int r = 0; r < R; r++) d[r] = row(slot, r)[ic];
  };
#pragma unroll
  for (int r = 0; r < R; r++) {
    G.pc[r] = row(pc_, r)[ic];
    G.po[r] = row(po_, r)[ic];
    G.fa[r] = row(a.fact, r)[ic];
    G.psx[r] = G.xix[r] = G.psz[r] = G.xiz[r] = T(0);
    if (ADJ) g[r] = row(a.grad + so, r)[ic];
  }
  T xc[4] = {T(0), T(0), T(0), T(0)};
  if (xs && h > 0) {
    const AxisCoef<T> cx = axis_coef(a.cpml + (int64_t)s * a.cstride, h, 0);
    const unsigned k = max(kx, 0);
    const T c0 = cx.bh(k), c1 = cx.ah(k), c2 = cx.b(k), c3 = cx.a(k);
    if (kx >= 0) {
      xc[0] = c0;
      xc[1] = c1;
      xc[2] = c2;
      xc[3] = c3;
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
      const int j = min(W.j0 + r, nz - 1);
      const T v0 = (a.psix_o + (int64_t)s * a.spx + (int64_t)j * (2 * h))[k];
      const T v1 = (a.xix_o + (int64_t)s * a.sxx + (int64_t)j * (2 * h + 2))[k];
      G.psx[r] = kx >= 0 ? v0 : T(0);
      G.xix[r] = kx >= 0 ? v1 : T(0);
    }
  }
  if (zs) {
#pragma unroll
    for (int r = 0; r < R; r++)
      if (W.kzr >> r & 1) {
        G.psz[r] = (a.psiz_o + (int64_t)s * a.spz + (int64_t)strip(r) * nx)[ic];
        G.xiz[r] = (a.xiz_o + (int64_t)s * a.sxz + (int64_t)strip(r) * nx)[ic];
      }
  }
  // levels of this shot: a forward one ends at nts, an adjoint one starts
  // there (from zero fields).  Tested after the loads above were issued, so
  // that they do not wait for nts.
  const int la = ADJ ? min(a.it, nts) : a.it;
  const int nl = ADJ ? la - (a.it - n) : min(n, nts - a.it + 1);
  if (nl <= 0 || nts <= a.act_min) return;
  // the history slot of forward level l is l - seg0 - 1 (none up to seg0)
  const int seg0 = a.dmode == 1 ? ((nts - 1) / a.S) * a.S : a.dmode == 2 ? a.cbase : a.it + n;
  if (ADJ) {
    fetch(d0, la);
    fetch(d1, la - 1);
  }
  // (loaded here: a load in the level loop would wait for the wave's stores)
  const int64_t otr = a.pt.off_tr[s];
  level_points<T, R, ADJ>(a, L, W, s, nts, X0, la, nl);
  if (threadIdx.x <= H) {
    const int j = Z0 - 1 + (int)threadIdx.x;
    int kz = -1;
    if (j >= 0 && j < h) kz = j;
    else if (j >= nz - h - 1 && j <= nz - 2) kz = j + 1 - nz + 2 * h;
    const AxisCoef<T> cz = axis_coef(a.cpml + (int64_t)s * a.cstride, h, 1);
    T *q = L.cz[threadIdx.x];
    q[0] = kz >= 0 ? cz.bh(kz) : T(0);
    q[1] = kz >= 0 ? cz.ah(kz) : T(0);
    q[2] = kz >= 0 ? cz.b(kz) : T(0);
    q[3] = kz >= 0 ? cz.a(kz) : T(0);
  }

  auto level = [&](int m, T *dv) {
    opaque(W.j0);
    opaque(W.rows);
    opaque(W.jin);
    opaque(W.kzr);
    opaque(W.xzr);
    opaque(W.imask);
    opaque(W.rmask);
    const int l = ADJ ? la - m : la + m;
    const int p = m & 1;
    L.first[p][W.w][W.lane] = G.pc[0];
    L.last[p][W.w][W.lane] = G.pc[R - 1];
    if (zs) L.lastz[p][W.w][W.lane] = G.psz[R - 1];
    __syncthreads();
    // (the first and last wave read rows of their own: the window's side)
    const T up = L.last[p][W.w > 0 ? W.w - 1 : 0][W.lane];
    const T dn = L.first[p][W.w < NW - 1 ? W.w + 1 : NW - 1][W.lane];
    const T zup = zs ? L.lastz[p][W.w > 0 ? W.w - 1 : 0][W.lane] : T(0);
    T dval[R];
    if (xs) cd2d_n_level<T, R, NW, ADJ, true, true>(a, L, W, kx, xc, up, dn, zup, G, dval);
    else if (zs) cd2d_n_level<T, R, NW, ADJ, false, true>(a, L, W, kx, xc, up, dn, zup, G, dval);
    else cd2d_n_level<T, R, NW, ADJ, false, false>(a, L, W, kx, xc, up, dn, zup, G, dval);
    if (W.imask | W.rmask) {
#pragma unroll
      for (int r = 0; r < R; r++) {
        if (W.imask >> r & 1) {
          T inj = 0;
          const T before = G.pc[r];      // of an edge cell: its level before last
          level_inject<T, R, ADJ>(a, L, W, s, nts, r, m, l, G.fa[r], G.pc[r], inj);
          if (!ADJ) {
            const bool interior = W.i >= 1 && W.i <= nx - 2 && (W.jin >> r & 1);
            dval[r] = interior ? dval[r] + inj : (before - T(2) * G.po[r]) + G.pc[r];
          }
        }
        if (!ADJ && (W.rmask & W.rows) >> r & 1 && W.own)
          level_record<T, R>(a, L, W, nts, r, a.traces + otr + (l - 1), G.pc[r]);
      }
    }
    if constexpr (ADJ) {
#pragma unroll
      for (int r = 0; r < R; r++) g[r] = g[r] + G.pc[r] * dv[r];
      fetch(dv, l - 2);
    } else {
      if (l > seg0 && W.own) {
        T *D = a.dbuf + (int64_t)(l - seg0 - 1) * a.dslot + so;
#pragma unroll
        for (int r = 0; r < R; r++)
          if (W.rows >> r & 1) (D + (int64_t)(W.j0 + r) * nx)[ic] = dval[r];
      }
    }
  };
  if constexpr (ADJ) {
    for (int m = 0; m < nl; m += 2) {
      level(m, d0);
      if (m + 1 < nl) level(m + 1, d1);
    }
  } else {
#pragma clang loop unroll(disable)
    for (int m = 0; m < nl; m++) level(m, d0);
  }

  if (!W.own) return;
#pragma unroll
  for (int r = 0; r < R; r++) {
    if (!(W.rows >> r & 1)) continue;
    const int64_t j = W.j0 + r, o = so + j * nx;
    (a.pnew + o)[ic] = G.pc[r];
    if (n > 1) (A.pnew0 + o)[ic] = G.po[r];
    if (ADJ) (a.grad + o)[ic] = g[r];
    if (kx >= 0) {
      (a.psix_n + (int64_t)s * a.spx + j * (2 * h))[(unsigned)kx] = G.psx[r];
      (a.xix + (int64_t)s * a.sxx + j * (2 * h + 2))[(unsigned)kx] = G.xix[r];
    }
    if (W.kzr >> r & 1) {
      (a.psiz_n + (int64_t)s * a.spz + (int64_t)strip(r) * nx)[ic] = G.psz[r];
      (a.xiz + (int64_t)s * a.sxz + (int64_t)strip(r) * nx)[ic] = G.xiz[r];
    }
  }
}

// grad += adjcur * D for the first step of a segment (the other steps are
// fused into the adjoint stencil).
template <typename T>
__global__ void cd2d_correlate_kernel(T *grad, const T *adj, const T *d, int64_t N, const int *nt_shot, int cbase) {
  const int s = blockIdx.y;
  if (nt_shot[s] <= cbase) return;
  const int64_t so = (int64_t)s * N;
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < N; q += (int64_t)gridDim.x * blockDim.x)
    grad[so + q] += adj[so + q] * d[so + q];
}

template <typename T>
class Cd2dEngine final : public Engine {
 public:
  explicit Cd2dEngine(PlanCore &core) : c_(core) {
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
    // rows per thread (1, 2 or 4) and the interior-tile path of
    // cd2d_step_kernel, which the environment picks (one level per launch)
    if (const char *v = std::getenv("SWX_CD2D_ROWS")) {
      const int r = std::atoi(v);
      SWX_REQUIRE(r == 1 || r == 2 || r == 4, SWX_EINVAL, "SWX_CD2D_ROWS must be 1, 2 or 4");
      rows_ = r;
      steps_env_ = 1;
    }
    if (const char *v = std::getenv("SWX_CD2D_LEAN")) lean_ = std::atoi(v) != 0;
    // most levels per launch (1: cd2d_step_kernel, else cd2d_stepn_kernel) and
    // window shape of the latter (10 x adjoint + forward)
    if (const char *v = std::getenv("SWX_CD2D_STEPS")) {
      steps_env_ = std::atoi(v);
      SWX_REQUIRE(steps_env_ >= 1 && steps_env_ <= SN_MAX, SWX_EINVAL, "SWX_CD2D_STEPS must be 1 .. 8");
    }
    if (const char *v = std::getenv("SWX_CD2D_SHAPE")) {
      shape_env_ = std::atoi(v);
      const int f = shape_env_ % 10, b = shape_env_ / 10;
      SWX_REQUIRE(shape_env_ >= 0 && f <= 2 && b <= 2 && !(b == 0) && !(f == 0 && sizeof(T) == 8) &&
                      !(b == 1 && sizeof(T) == 8), SWX_EINVAL, "SWX_CD2D_SHAPE names a shape that is not built");
    }
    const size_t e = sizeof(T);
    fact_.alloc(N_ * e);
    // forward state: four pressure levels and the C-PML memory variables of
    // three: a launch reads the two last levels and writes its own two last
    // ones to the other slots, so that it never overwrites what a
    // neighbouring block still reads (cd2d_stepn_kernel)
    p_.alloc(4 * ns_ * N_ * e);
    psix_.alloc(std::max<int64_t>(3 * ns_ * spx_, 1) * e);
    psiz_.alloc(std::max<int64_t>(3 * ns_ * spz_, 1) * e);
    xix_.alloc(std::max<int64_t>(3 * ns_ * sxx_, 1) * e);
    xiz_.alloc(std::max<int64_t>(3 * ns_ * sxz_, 1) * e);
    cpml_.alloc((int64_t)ns_ * cstride_ * e);
    state_bytes_ = fact_.bytes() + p_.bytes() + psix_.bytes() + psiz_.bytes() + xix_.bytes() + xiz_.bytes();
    if (d.gradient) {
      a_.alloc(4 * ns_ * N_ * e);
      // adjoint state: the same level layout as the forward state
      apsix_.alloc(psix_.bytes());
      apsiz_.alloc(psiz_.bytes());
      axix_.alloc(xix_.bytes());
      axiz_.alloc(xiz_.bytes());
      grad_.alloc(ns_ * N_ * e);
      gout_.alloc(ns_ * N_ * e);
      state_bytes_ += a_.bytes() + apsix_.bytes() + apsiz_.bytes() + axix_.bytes() +
                      axiz_.bytes() + grad_.bytes() + gout_.bytes();
      const int64_t slot = ns_ * N_ * (int64_t)e;
      ck_bytes_one_ = (2 * N_ + spx_ + spz_ + sxx_ + sxz_) * ns_ * (int64_t)e;
      int64_t avail = (int64_t)c_.budget - state_bytes_;
      S_ = choose_segment(d.nt_max, d.check_freq, slot, ck_bytes_one_, avail);
      K_ = (int)ceil_div(d.nt_max, S_);
      dbuf_.alloc((int64_t)S_ * slot);
      nck_ = std::max(K_ - 2, 0);
      ck_.alloc(std::max<int64_t>(nck_ * ck_bytes_one_, 1));
    }
    zero_forward_state();
  }

  void set_model(int nfields, const void *const *fields) override {
    SWX_REQUIRE(nfields == 1 && fields[0], SWX_EINVAL, "acoustic CD expects one model field (fact)");
    SWX_HIP(hipMemcpyAsync(fact_.get(), fields[0], N_ * sizeof(T), hipMemcpyHostToDevice, c_.stream));
    SWX_HIP(hipStreamSynchronize(c_.stream));
    model_set_ = true;
  }

  void on_shots_set(int nshots, const swx_shot_desc *shots) override {
    std::vector<T> hc((size_t)nshots * cstride_);
    const int la = 2 * h_ + 2, lh = 2 * h_;
    for (int s = 0; s < nshots; s++) {
      T *dst = hc.data() + (size_t)s * cstride_;
      for (int ax = 0; ax < 2; ax++) {
        const int len[4] = {la, lh, la, lh};
        T *p = dst + ax * (8 * h_ + 4);
        for (int k = 0; k < 4; k++) {
          const T *src = static_cast<const T *>(shots[s].cpml[ax][k]);
          SWX_REQUIRE(src || len[k] == 0, SWX_EINVAL, "missing C-PML coefficient array");
          if (len[k]) std::memcpy(p, src, sizeof(T) * len[k]);
          p += len[k];
        }
      }
      SWX_REQUIRE(shots[s].nt <= c_.d.nt_max, SWX_EINVAL, "shot nt exceeds nt_max");
    }
    SWX_HIP(hipMemcpyAsync(cpml_.get(), hc.data(), hc.size() * sizeof(T), hipMemcpyHostToDevice, c_.stream));
    SWX_HIP(hipStreamSynchronize(c_.stream));
    nsh_ = nshots;
    nt_ = c_.pts.nt;
    ntmax_ = *std::max_element(nt_.begin(), nt_.end());
  }

  void forward(bool save) override {
    SWX_REQUIRE(model_set_, SWX_ESTATE, "swx_set_model must be called before running");
    zero_forward_state();
    T *tr = c_.pts.d_traces.as<T>();
    choose_steps();
    for (int it = 1; it <= ntmax_;) {
      progress("forward step", it, ntmax_);
      // a launch ends at the levels whose state is kept: checkpoints (its two
      // last levels) and snapshots
      int end = ntmax_;
      if (save) end = std::min<int64_t>(end, ceil_div(it, S_) * (int64_t)S_);
      if (c_.snap_every > 0) end = std::min<int64_t>(end, ceil_div(it, c_.snap_every) * (int64_t)c_.snap_every);
      const int n = levels(end - it + 1);
      step_fwd(it, n, /*act_min=*/0, save ? 1 : 0, /*cbase=*/0, tr);
      it += n;
      const int l = it - 1;
      take_snapshots(c_, *this, l);
      if (save && l % S_ == 0) {
        const int k = l / S_;
        if (k >= 1 && k <= K_ - 2) save_ckpt(k);
      }
    }
  }

  // "pcur" (acou_forward.jl:55-57): the level stepped last
  int snap_fields(int, int s, SnapPiece *out) const override {
    out[0] = {P(f_.cur) + (int64_t)s * N_, (int64_t)(N_ * sizeof(T)), (int64_t)(N_ * sizeof(T)), 1};
    return 1;
  }

  void adjoint(bool per_shot) override {
    (void)per_shot;
    b_ = Pos{};
    SWX_HIP(hipMemsetAsync(a_.get(), 0, a_.bytes(), c_.stream));
    SWX_HIP(hipMemsetAsync(apsix_.get(), 0, apsix_.bytes(), c_.stream));
    SWX_HIP(hipMemsetAsync(apsiz_.get(), 0, apsiz_.bytes(), c_.stream));
    SWX_HIP(hipMemsetAsync(axix_.get(), 0, axix_.bytes(), c_.stream));
    SWX_HIP(hipMemsetAsync(axiz_.get(), 0, axiz_.bytes(), c_.stream));
    SWX_HIP(hipMemsetAsync(grad_.get(), 0, grad_.bytes(), c_.stream));
    const int Kmax = (int)ceil_div(ntmax_, S_);
    for (int k = Kmax - 1; k >= 0; k--) {
      progress("adjoint segment", Kmax - k, Kmax);
      const int cb = k * S_;
      // replay for shots whose segment k is not their last one
      bool need = false;
      for (int s = 0; s < nsh_; s++) need |= nt_[s] > cb + S_;
      if (need) {
        restore_ckpt(k);
        for (int it = cb + 1; it <= cb + S_;) {
          const int n = levels(cb + S_ - it + 1);
          step_fwd(it, n, cb + S_, 2, cb, nullptr);
          it += n;
        }
      }
      const int top = std::min(cb + S_, ntmax_);
      for (int it = top; it >= cb + 1;) {
        const int n = levels(it - cb);
        step_adj(it, n, cb);
        it -= n;
      }
      if (steps_ == 1) {
        // correlation of the first step of the segment (cd2d_stepn_kernel
        // correlates every level that it steps)
        dim3 g((unsigned)std::min<int64_t>(ceil_div(N_, 256), 1024), nsh_);
        cd2d_correlate_kernel<T><<<g, 256, 0, c_.stream>>>(grad_.as<T>(), A(b_.cur), dbuf_.as<T>(), N_,
                                                            c_.pts.d_nt.as<int>(), cb);
        SWX_HIP(hipGetLastError());
      }
    }
    const T scale = T(1.0 / (c_.d.dt * c_.d.dt));
    dim3 g((unsigned)std::min<int64_t>(ceil_div(N_, 256), 4096));
    reduce_shots<T><<<g, 256, 0, c_.stream>>>(gout_.as<T>(), grad_.as<T>(), N_, nsh_, scale, per_shot ? 1 : 0);
    SWX_HIP(hipGetLastError());
  }

  void copy_grad(void *host, bool per_shot) override {
    const size_t bytes = (per_shot ? (size_t)nsh_ : 1) * N_ * sizeof(T);
    SWX_HIP(hipMemcpy(host, gout_.get(), bytes, hipMemcpyDeviceToHost));
  }

  int64_t bytes_state() const override { return state_bytes_; }
  int64_t bytes_checkpoints() const override { return ck_.bytes(); }
  int64_t bytes_replay() const override { return dbuf_.bytes(); }
  int segment() const override { return S_; }
  // rows per thread of the one-level kernel, or window shapes of the n-level
  // one (10 x adjoint + forward); most levels per launch, 10 x adjoint +
  // forward / replay
  void variants(int32_t v[2]) const override {
    v[0] = steps_ == 1 ? rows_ : 10 * shape_[1] + shape_[0];
    v[1] = 11 * steps_;
  }

 private:
  // Slots of the levels of a state: the last level is in pressure slot cur,
  // the one before it in cur - 1 (mod 4), the memory variables in buffer mv.
  struct Pos {
    int cur = 0, mv = 0;
  };
  void advance(Pos &p, int n) const {
    p.cur = (p.cur + std::min(n, 2)) & 3;
    p.mv = (p.mv + 1) % 3;
  }
  T *P(int k) const { return p_.as<T>() + (int64_t)(k & 3) * ns_ * N_; }
  T *PSX(int k) const { return psix_.as<T>() + (int64_t)(k % 3) * ns_ * spx_; }
  T *PSZ(int k) const { return psiz_.as<T>() + (int64_t)(k % 3) * ns_ * spz_; }
  T *XIX(int k) const { return xix_.as<T>() + (int64_t)(k % 3) * ns_ * sxx_; }
  T *XIZ(int k) const { return xiz_.as<T>() + (int64_t)(k % 3) * ns_ * sxz_; }
  T *A(int k) const { return a_.as<T>() + (int64_t)(k & 3) * ns_ * N_; }
  T *APSX(int k) const { return apsix_.as<T>() + (int64_t)(k % 3) * ns_ * spx_; }
  T *APSZ(int k) const { return apsiz_.as<T>() + (int64_t)(k % 3) * ns_ * spz_; }
  T *AXIX(int k) const { return axix_.as<T>() + (int64_t)(k % 3) * ns_ * sxx_; }
  T *AXIZ(int k) const { return axiz_.as<T>() + (int64_t)(k % 3) * ns_ * sxz_; }

  // Levels of the next launch when `left` remain: launches of nearly equal
  // size, none above steps_.
  int levels(int left) const {
    const int launches = (int)ceil_div(left, steps_);
    return (int)ceil_div(left, launches);
  }

  // Windows of a launch of n levels over the batch, H rows each.
  int64_t windows(int H, int n) const {
    return std::max<int64_t>(ceil_div(nx_ - 2 * n, TX - 2 * n), 1) *
           std::max<int64_t>(ceil_div(nz_ - 2 * n, H - 2 * n), 1) * nsh_;
  }

  // Levels per launch: as many as a window can step, since a launch costs 5-7
  // us (loads, stores, the gap to the next one) whatever it steps and a level
  // 1-3 us: 8 levels are the fastest everywhere from 121 x 101 cells to
  // 4 x 2000 x 1000 (4 levels: 1.1 to 1.6 times as long per level).
  // Window shape, us per level measured forward / adjoint:
  //   2 (16 waves, 2 rows per thread, 32 rows): the shortest level, for grids
  //     that leave CUs idle.  f32 201 x 151: 2.1 / 1.5 against 2.5 / 2.1 in
  //     shape 1; 500 x 400 (264 windows): 2.2 / 1.7 against 2.5 / 2.1;
  //     4 x 300 x 250 (360 windows): 2.8 / 2.7 against 2.5 / 2.3.
  //   1 (16 waves, 4 rows, 64 rows): less work on cells that the neighbours
  //     step too.  f32 700 x 700 (225 windows): 2.6 / 2.3 against 3.6 / 4.4
  //     in shape 0; f64 16 x 600 x 400 forward: 15.7 against 23.8 in shape 2.
  //     The f64 adjoint spills in it (37.8 against 25.6) and stays in shape 2.
  //   0 (8 waves, 8 rows, 64 rows): f32 forward with more windows of 64 rows
  //     than CUs, two blocks to a CU: 16 x 600 x 400: 9.6 against 11.3 in
  //     shape 1; the f32 adjoint spills (19.7 against 11.6).
  void choose_steps() {
    steps_ = steps_env_ ? steps_env_ : SN_MAX;
    const bool small = windows(32, SN_MAX) <= 300, many = windows(64, SN_MAX) > 256;
    shape_[0] = small ? 2 : many && sizeof(T) == 4 ? 0 : 1;
    shape_[1] = small || sizeof(T) == 8 ? 2 : 1;
    if (shape_env_ >= 0) {
      shape_[0] = shape_env_ % 10;
      shape_[1] = shape_env_ / 10;
    }
  }

  void zero_forward_state() {
    f_ = Pos{};
    SWX_HIP(hipMemsetAsync(p_.get(), 0, p_.bytes(), c_.stream));
    SWX_HIP(hipMemsetAsync(psix_.get(), 0, psix_.bytes(), c_.stream));
    SWX_HIP(hipMemsetAsync(psiz_.get(), 0, psiz_.bytes(), c_.stream));
    SWX_HIP(hipMemsetAsync(xix_.get(), 0, xix_.bytes(), c_.stream));
    SWX_HIP(hipMemsetAsync(xiz_.get(), 0, xiz_.bytes(), c_.stream));
  }

  Cd2dStepArgs<T> base_args(int it) const {
    Cd2dStepArgs<T> a{};
    a.nx = nx_; a.nz = nz_; a.h = h_; a.N = N_;
    a.idx = T(1.0 / c_.d.h[0]);
    a.idz = T(1.0 / c_.d.h[1]);
    a.idx2 = a.idx * a.idx;
    a.idz2 = a.idz * a.idz;
    a.fact = fact_.as<T>();
    a.spx = spx_; a.spz = spz_; a.sxx = sxx_; a.sxz = sxz_;
    a.cpml = cpml_.as<T>(); a.cstride = cstride_;
    a.nt_shot = c_.pts.d_nt.as<int>();
    a.it = it;
    a.dbuf = dbuf_.as<T>(); a.dslot = (int64_t)ns_ * N_; a.S = S_ > 0 ? S_ : 1;
    a.pt = view(c_.pts);
    a.srctf = c_.pts.d_srctf.as<T>();
    return a;
  }

  // e0 / e1 (nullable): events the dispatch records at the kernel's start
  // and end
  template <int R>
  void launch_rows(Cd2dStepArgs<T> a, hipEvent_t e0 = nullptr, hipEvent_t e1 = nullptr) {
    a.nbx = (int)ceil_div(nx_, TX);
    a.nby = (int)ceil_div(nz_, TZ * R);
    const unsigned nb = (unsigned)((int64_t)a.nbx * a.nby * nsh_);
    hipExtLaunchKernelGGL(cd2d_step_kernel<T, R>, dim3(nb), dim3(TX, TZ), 0, c_.stream, e0, e1, 0, a);
  }

  // A launch here lasts about 9 us, so event packets around it would add a
  // fifth to the measured time: the per-launch timing uses the events the
  // dispatch itself records.
  void launch(Cd2dStepArgs<T> a) {
    a.lean = lean_ ? 1 : 0;
    hipEvent_t e0, e1;
    c_.ktimer.dispatch_events(a.corr ? 1 : 0, &e0, &e1);
    if (rows_ == 4) launch_rows<4>(a, e0, e1);
    else if (rows_ == 1) launch_rows<1>(a, e0, e1);
    else launch_rows<2>(a, e0, e1);
    SWX_HIP(hipGetLastError());
  }

  Cd2dStepArgs<T> fwd_args(int it, int act_min, int dmode, int cbase, T *traces) const {
    Cd2dStepArgs<T> a = base_args(it);
    a.pold = P(f_.cur + 3); a.pcur = P(f_.cur); a.pnew = P(f_.cur + 1);
    a.psix_o = PSX(f_.mv); a.psix_n = PSX(f_.mv + 1);
    a.psiz_o = PSZ(f_.mv); a.psiz_n = PSZ(f_.mv + 1);
    a.xix_o = XIX(f_.mv); a.xix = XIX(f_.mv + 1);
    a.xiz_o = XIZ(f_.mv); a.xiz = XIZ(f_.mv + 1);
    a.act_min = act_min;
    a.dmode = c_.d.gradient ? dmode : 0;
    a.cbase = cbase;
    a.corr = 0;
    a.traces = traces;
    return a;
  }

  template <int R, int NW, bool ADJ>
  void launch_shape(Cd2dStepNArgs<T> &A) {
    constexpr int H = NW * R;
    A.a.nbx = (int)std::max<int64_t>(ceil_div(nx_ - 2 * A.n, TX - 2 * A.n), 1);
    A.a.nby = (int)std::max<int64_t>(ceil_div(nz_ - 2 * A.n, H - 2 * A.n), 1);
    hipEvent_t e0, e1;
    c_.ktimer.dispatch_events(ADJ ? 1 : 0, &e0, &e1);
    hipExtLaunchKernelGGL((cd2d_stepn_kernel<T, R, NW, ADJ>), dim3((unsigned)((int64_t)A.a.nbx * A.a.nby * nsh_)),
                          dim3(NW * TX), 0, c_.stream, e0, e1, 0, A);
    SWX_HIP(hipGetLastError());
  }
  template <bool ADJ>
  void launch_stepn(const Cd2dStepArgs<T> &a, T *pnew0, int n) {
    Cd2dStepNArgs<T> A;
    A.a = a;
    A.pnew0 = pnew0;
    A.n = n;
    const int shape = shape_[ADJ];
    if (shape == 2) {
      launch_shape<2, 16, ADJ>(A);
      return;
    }
    if constexpr (sizeof(T) == 4 || !ADJ) {
      if (shape == 1) {
        launch_shape<4, 16, ADJ>(A);
        return;
      }
    }
    if constexpr (sizeof(T) == 4 && !ADJ) launch_shape<8, 8, ADJ>(A);
  }

  // forward / replay levels it .. it+n-1
  void step_fwd(int it, int n, int act_min, int dmode, int cbase, T *traces) {
    Cd2dStepArgs<T> a = fwd_args(it, act_min, dmode, cbase, traces);
    if (steps_ == 1) {
      launch(a);
    } else {
      T *older = a.pnew;
      if (n > 1) a.pnew = P(f_.cur + 2);
      launch_stepn<false>(a, older, n);
    }
    advance(f_, n);
  }

  Cd2dStepArgs<T> adj_args(int it, int cbase) const {
    Cd2dStepArgs<T> a = base_args(it);
    a.pold = A(b_.cur + 3); a.pcur = A(b_.cur); a.pnew = A(b_.cur + 1);
    a.psix_o = APSX(b_.mv); a.psix_n = APSX(b_.mv + 1);
    a.psiz_o = APSZ(b_.mv); a.psiz_n = APSZ(b_.mv + 1);
    a.xix_o = AXIX(b_.mv); a.xix = AXIX(b_.mv + 1);
    a.xiz_o = AXIZ(b_.mv); a.xiz = AXIZ(b_.mv + 1);
    a.act_min = 0;
    a.dmode = 0;
    a.cbase = cbase;
    a.grad = grad_.as<T>();
    a.corr = 1;
    a.corr_lim = cbase + S_;
    a.res = c_.pts.d_res.as<T>();
    return a;
  }
  // adjoint levels it .. it-n+1
  void step_adj(int it, int n, int cbase) {
    Cd2dStepArgs<T> a = adj_args(it, cbase);
    if (steps_ == 1) {
      launch(a);
    } else {
      T *older = a.pnew;
      if (n > 1) a.pnew = A(b_.cur + 2);
      launch_stepn<true>(a, older, n);
    }
    advance(b_, n);
  }

  // checkpoint layout (all shots): p^{c-1} | p^c | psi_x | psi_z | xi_x | xi_z
  void ckpt_copy(int k, bool save) {
    const int64_t e = sizeof(T);
    char *base = ck_.as<char>() + (int64_t)(k - 1) * ck_bytes_one_;
    const int64_t fb = (int64_t)ns_ * N_ * e;
    struct Part { void *dev; int64_t bytes; };
    Part parts[6] = {
        {P(f_.cur + 3), fb},
        {P(f_.cur), fb},
        {PSX(f_.mv), ns_ * spx_ * e},
        {PSZ(f_.mv), ns_ * spz_ * e},
        {XIX(f_.mv), ns_ * sxx_ * e},
        {XIZ(f_.mv), ns_ * sxz_ * e},
    };
    int64_t off = 0;
    for (auto &pt : parts) {
      if (pt.bytes) {
        if (save)
          SWX_HIP(hipMemcpyAsync(base + off, pt.dev, pt.bytes, hipMemcpyDeviceToDevice, c_.stream));
        else
          SWX_HIP(hipMemcpyAsync(pt.dev, base + off, pt.bytes, hipMemcpyDeviceToDevice, c_.stream));
      }
      off += pt.bytes;
    }
  }
  void save_ckpt(int k) { ckpt_copy(k, true); }
  void restore_ckpt(int k) {
    if (k == 0) {
      zero_forward_state();
    } else {
      ckpt_copy(k, false);
    }
  }

  PlanCore &c_;
  int nx_, nz_, h_, ns_;
  int64_t N_, spx_, spz_, sxx_, sxz_;
  int cstride_;
  int rows_ = 2;         // rows per thread of cd2d_step_kernel
  int steps_ = 1, shape_[2] = {0, 0};     // most levels per launch, block shapes (forward, adjoint)
  int steps_env_ = 0, shape_env_ = -1;    // pinned by the environment (0, -1: not)
  Pos f_, b_;                             // forward and adjoint state
  bool lean_ = true;
  DevBuf fact_, p_, psix_, psiz_, xix_, xiz_, cpml_;
  DevBuf a_, apsix_, apsiz_, axix_, axiz_, grad_, gout_;
  DevBuf dbuf_, ck_;
  int64_t ck_bytes_one_ = 0, state_bytes_ = 0;
  int S_ = 1, K_ = 1, nck_ = 0;
  int nsh_ = 0, ntmax_ = 0;
  std::vector<int> nt_;
  bool model_set_ = false;
};

}  // namespace

std::unique_ptr<Engine> make_acoustic_cd2d(PlanCore &core) {
  if (core.d.dtype == SWX_F32) return std::make_unique<Cd2dEngine<float>>(core);
  return std::make_unique<Cd2dEngine<double>>(core);
}

}  // namespace swx

// ---------------------------------------------------------------------------
// swx_forward_noalloc: the forward of one shot without any device allocation
// ---------------------------------------------------------------------------
// Every byte of device memory the call uses (model, three time levels, C-PML
// memory variables and coefficients, point tables, source time function and
// traces) is carved out of this array.  Each GPU the library runs on holds
// its own copy until the process ends; calls on one GPU share it.
static __device__ __align__(256) unsigned char scratch[SWX_NOALLOC_SCRATCH_BYTES];

namespace swx {
namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch_dev[kMaxDevices] = {};

// Device address of `scratch` on the current device `dev`, looked up once
// per device.  The host-side name `scratch` is not a device address.
void *scratch_on(int dev) {
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  SWX_REQUIRE(dev >= 0 && dev < kMaxDevices, SWX_EINVAL, "invalid device ordinal");
  if (!g_scratch_dev[dev]) {
    void *ptr = nullptr;
    SWX_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    SWX_REQUIRE(ptr != nullptr, SWX_EHIP, "hipGetSymbolAddress(scratch) returned no address");
    g_scratch_dev[dev] = ptr;
  }
  return g_scratch_dev[dev];
}

__global__ void zero_words(uint32_t *p, int64_t n) {
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < n; q += (int64_t)gridDim.x * blockDim.x)
    p[q] = 0u;
}

// Offsets of the pieces in the scratch array, each aligned to 256 bytes.
struct Carve {
  size_t off = 0;
  size_t take(size_t bytes) {
    off = (off + 255) & ~size_t(255);
    const size_t o = off;
    off += bytes;
    return o;
  }
};

template <typename T>
void forward_noalloc(const swx_plan_desc &d, const T *fact, const swx_shot_desc &shot, T *traces_host) {
  const int nx = (int)d.n[0], nz = (int)d.n[1], h = d.halo;
  const int64_t N = (int64_t)nx * nz;
  const int64_t spx = (int64_t)2 * h * nz, spz = (int64_t)nx * 2 * h;
  const int64_t sxx = (int64_t)(2 * h + 2) * nz, sxz = (int64_t)nx * (2 * h + 2);
  const int cstride = 2 * (8 * h + 4);
  HostPointTables t;
  host_point_tables(t, 2, d.n, 1, &shot);
  const std::vector<T> cp = pack_cpml<T>(1, &shot, 2, h);
  const int nt = shot.nt;
  // the pieces copied from the host come first, the ones cleared on the
  // device after them
  Carve cv;
  const size_t o_fact = cv.take(N * sizeof(T));
  const size_t o_cpml = cv.take(cp.size() * sizeof(T));
  const size_t o_nt = cv.take(sizeof(int));
  const size_t o_offtf = cv.take(sizeof(int64_t)), o_offtr = cv.take(sizeof(int64_t));
  const size_t o_usrc_off = cv.take(t.usrc_off.size() * sizeof(int));
  const size_t o_usrc_cell = cv.take(t.usrc_cell.size() * sizeof(int64_t));
  const size_t o_usrc_ptr = cv.take(t.usrc_ptr.size() * sizeof(int));
  const size_t o_usrc_list = cv.take(t.usrc_list.size() * sizeof(int));
  const size_t o_urec_off = cv.take(t.urec_off.size() * sizeof(int));
  const size_t o_urec_cell = cv.take(t.urec_cell.size() * sizeof(int64_t));
  const size_t o_urec_ptr = cv.take(t.urec_ptr.size() * sizeof(int));
  const size_t o_urec_list = cv.take(t.urec_list.size() * sizeof(int));
  const size_t o_rec_off = cv.take(t.rec_off.size() * sizeof(int));
  const size_t o_rec_cell = cv.take(t.rec_cell.size() * sizeof(int64_t));
  const size_t o_srow = cv.take(t.srow.size() * sizeof(int));
  const size_t o_rrow = cv.take(t.rrow.size() * sizeof(int));
  const size_t o_tf = cv.take((size_t)t.total_tf * sizeof(T));
  const size_t copy_end = cv.take(0);
  const size_t o_p = cv.take((size_t)3 * N * sizeof(T));
  const size_t o_psix = cv.take((size_t)2 * spx * sizeof(T)), o_psiz = cv.take((size_t)2 * spz * sizeof(T));
  const size_t o_xix = cv.take((size_t)sxx * sizeof(T)), o_xiz = cv.take((size_t)sxz * sizeof(T));
  const size_t o_tr = cv.take((size_t)t.total_tr * sizeof(T));
  const size_t total = cv.take(0);
  SWX_REQUIRE(total <= SWX_NOALLOC_SCRATCH_BYTES, SWX_ENOMEM,
              "swx_forward_noalloc: the shot needs " + std::to_string(total) + " bytes of device memory, more than "
              "the " + std::to_string((size_t)SWX_NOALLOC_SCRATCH_BYTES) + "-byte scratch array");

  std::vector<char> stage(copy_end);
  auto put = [&](size_t o, const void *src, size_t bytes) {
    if (bytes) std::memcpy(stage.data() + o, src, bytes);
  };
  const int64_t zero64 = 0;
  put(o_fact, fact, N * sizeof(T));
  put(o_cpml, cp.data(), cp.size() * sizeof(T));
  put(o_nt, &nt, sizeof(int));
  put(o_offtf, &zero64, sizeof(int64_t));
  put(o_offtr, &zero64, sizeof(int64_t));
  put(o_usrc_off, t.usrc_off.data(), t.usrc_off.size() * sizeof(int));
  put(o_usrc_cell, t.usrc_cell.data(), t.usrc_cell.size() * sizeof(int64_t));
  put(o_usrc_ptr, t.usrc_ptr.data(), t.usrc_ptr.size() * sizeof(int));
  put(o_usrc_list, t.usrc_list.data(), t.usrc_list.size() * sizeof(int));
  put(o_urec_off, t.urec_off.data(), t.urec_off.size() * sizeof(int));
  put(o_urec_cell, t.urec_cell.data(), t.urec_cell.size() * sizeof(int64_t));
  put(o_urec_ptr, t.urec_ptr.data(), t.urec_ptr.size() * sizeof(int));
  put(o_urec_list, t.urec_list.data(), t.urec_list.size() * sizeof(int));
  put(o_rec_off, t.rec_off.data(), t.rec_off.size() * sizeof(int));
  put(o_rec_cell, t.rec_cell.data(), t.rec_cell.size() * sizeof(int64_t));
  put(o_srow, t.srow.data(), t.srow.size() * sizeof(int));
  put(o_rrow, t.rrow.data(), t.rrow.size() * sizeof(int));
  put(o_tf, shot.srctf, (size_t)t.total_tf * sizeof(T));

  char *base = static_cast<char *>(scratch_on(d.device));
  const hipStream_t stream = nullptr;
  SWX_HIP(hipMemcpyAsync(base, stage.data(), copy_end, hipMemcpyHostToDevice, stream));
  // the time levels, memory variables and traces start at zero
  const int64_t words = (int64_t)(total - copy_end) / 4;
  zero_words<<<(unsigned)std::min<int64_t>(ceil_div(words, 256), 2048), 256, 0, stream>>>(
      reinterpret_cast<uint32_t *>(base + copy_end), words);
  SWX_HIP(hipGetLastError());

  auto at = [&](size_t o) { return base + o; };
  PointArgsView pv{reinterpret_cast<const int *>(at(o_nt)), reinterpret_cast<const int64_t *>(at(o_offtf)),
                   reinterpret_cast<const int64_t *>(at(o_offtr)), reinterpret_cast<const int *>(at(o_usrc_off)),
                   reinterpret_cast<const int64_t *>(at(o_usrc_cell)), reinterpret_cast<const int *>(at(o_usrc_ptr)),
                   reinterpret_cast<const int *>(at(o_usrc_list)), reinterpret_cast<const int *>(at(o_urec_off)),
                   reinterpret_cast<const int64_t *>(at(o_urec_cell)), reinterpret_cast<const int *>(at(o_urec_ptr)),
                   reinterpret_cast<const int *>(at(o_urec_list)), reinterpret_cast<const int *>(at(o_rec_off)),
                   reinterpret_cast<const int64_t *>(at(o_rec_cell)), reinterpret_cast<const int *>(at(o_srow)),
                   reinterpret_cast<const int *>(at(o_rrow)), t.nrows};
  T *p = reinterpret_cast<T *>(at(o_p));
  T *psix = reinterpret_cast<T *>(at(o_psix));
  T *psiz = reinterpret_cast<T *>(at(o_psiz));
  T *tr = reinterpret_cast<T *>(at(o_tr));
  constexpr int R = 2;
  Cd2dStepArgs<T> a{};
  a.nx = nx; a.nz = nz; a.h = h; a.N = N;
  a.idx = T(1.0 / d.h[0]);
  a.idz = T(1.0 / d.h[1]);
  a.idx2 = a.idx * a.idx;
  a.idz2 = a.idz * a.idz;
  a.fact = reinterpret_cast<const T *>(at(o_fact));
  a.spx = spx; a.spz = spz; a.sxx = sxx; a.sxz = sxz;
  a.xix = reinterpret_cast<T *>(at(o_xix));
  a.xiz = reinterpret_cast<T *>(at(o_xiz));
  a.xix_o = a.xix;
  a.xiz_o = a.xiz;
  a.cpml = reinterpret_cast<const T *>(at(o_cpml)); a.cstride = cstride;
  a.nt_shot = pv.nt;
  a.S = 1;
  a.pt = pv;
  a.srctf = reinterpret_cast<const T *>(at(o_tf));
  a.traces = tr;
  a.lean = 1;
  a.nbx = (int)ceil_div(nx, TX);
  a.nby = (int)ceil_div(nz, TZ * R);
  const unsigned nb = (unsigned)((int64_t)a.nbx * a.nby);
  for (int it = 1; it <= nt; it++) {
    a.it = it;
    a.pold = p + (int64_t)mod3(it - 2) * N;
    a.pcur = p + (int64_t)mod3(it - 1) * N;
    a.pnew = p + (int64_t)mod3(it) * N;
    a.psix_o = psix + (int64_t)((it - 1) & 1) * spx;
    a.psix_n = psix + (int64_t)(it & 1) * spx;
    a.psiz_o = psiz + (int64_t)((it - 1) & 1) * spz;
    a.psiz_n = psiz + (int64_t)(it & 1) * spz;
    cd2d_step_kernel<T, R><<<nb, dim3(TX, TZ), 0, stream>>>(a);
    SWX_HIP(hipGetLastError());
  }
  SWX_HIP(hipMemcpyAsync(traces_host, tr, (size_t)t.total_tr * sizeof(T), hipMemcpyDeviceToHost, stream));
  SWX_HIP(hipStreamSynchronize(stream));
}

}  // namespace
}  // namespace swx

extern "C" int swx_forward_noalloc(const swx_plan_desc *desc, const void *fact, const swx_shot_desc *shot,
                                   void *traces) {
  using namespace swx;
  return guarded([&] {
    SWX_REQUIRE(desc && fact && shot && traces, SWX_EINVAL, "null argument");
    const swx_plan_desc &d = *desc;
    SWX_REQUIRE(d.physics == SWX_ACOUSTIC_CD && d.ndim == 2, SWX_EUNSUPPORTED,
                "swx_forward_noalloc runs 2D acoustic constant-density shots");
    validate_plan_desc(d);
    SWX_REQUIRE(shot->nt >= 1 && shot->nt <= d.nt_max, SWX_EINVAL, "shot nt must be in 1..nt_max");
    SWX_HIP(hipSetDevice(d.device));
    if (d.dtype == SWX_F32)
      forward_noalloc<float>(d, static_cast<const float *>(fact), *shot, static_cast<float *>(traces));
    else
      forward_noalloc<double>(d, static_cast<const double *>(fact), *shot, static_cast<double *>(traces));
  });
}
