// Points of a block that steps a 64-column window of registers by several
// levels per launch: the injected values of all its levels and the trace of
// every recorded cell, staged once in LDS.
#pragma once
#include "swx_device.hpp"

namespace swx {

constexpr int SN_MAX = 8;        // most levels per launch
constexpr int SN_SLOTS = 126;    // staged point values per level
constexpr int SN_RECS = 254;     // receivers whose traces are kept

// H rows of 64 columns
template <typename T, int H>
struct LevelPoints {
  short inj[H][64];            // staged values of a cell's points: slot + 1 and, above bit 7, their number;
                               // 0: no point, -1: not staged
  short rec[H][64];            // a cell's entries of col: first + 1 and, above bit 8, their number; 0, -1 alike
  T val[SN_MAX][SN_SLOTS];
  int col[SN_RECS];            // traces of the window's receivers
  int used, rused;             // slots and entries taken
};

// Window of a block and what its threads own.
struct LevelWin {
  int i, j0, w, lane;
  bool own;            // column owned
  int rows;            // rows of this wave owned (bit r: row r)
  int jin, kzr, xzr;   // rows inside the grid's z edges, with a psi_z / a xi_z
  int jg, jv;          // rows of the grid, of the z-staggered grid
  int imask, rmask;    // rows that hold injected points / receivers
};

// Injection of the level with index m (of the nl staged ones) and number l at
// row r: p += value (times the factor in the adjoint), in list order.
template <typename T, int R, bool ADJ, typename Args, typename Lds>
__device__ __forceinline__ void level_inject(const Args &a, const Lds &L, const LevelWin &W, int s, int nts, int r,
                                             int m, int l, T f, T &pnv, T &inj) {
  const int e = L.inj[W.w * R + r][W.lane];
  if (e == 0) return;
  auto add = [&](T v) {
    if (ADJ) {
      pnv += v * f;
    } else {
      pnv += v;
      inj += v;
    }
  };
  if (e > 0) {
    const T *v = L.val[m] + (e & 127) - 1;
#pragma clang loop unroll(disable)
    for (int k = 0; k < e >> 7; k++) add(v[k]);
    return;
  }
  const int *ptr = ADJ ? a.pt.urec_ptr : a.pt.usrc_ptr, *list = ADJ ? a.pt.urec_list : a.pt.usrc_list;
  const T *tf = (ADJ ? a.res + a.pt.off_tr[s] : a.srctf + a.pt.off_tf[s]) + (l - 1);
  const int j = W.j0 + r;
  const int u = find_point(ADJ ? a.pt.rrow : a.pt.srow, ADJ ? a.pt.urec_cell : a.pt.usrc_cell, a.pt.nrows, s, j,
                           (int64_t)j * a.nx + W.i);
#pragma clang loop unroll(disable)
  for (int k = ptr[u]; k < ptr[u + 1]; k++) add(tf[(int64_t)nts * list[k]]);
}

// Points of the wave's rows: the cells' entries in LDS, and (injected points)
// their values of the levels la, la + dir, .. (nl of them).
template <typename T, int R, bool ADJ, typename Args, typename Lds>
__device__ __forceinline__ void level_points(const Args &a, Lds &L, LevelWin &W, int s, int nts, int X0, int la,
                                             int nl) {
  constexpr int TX = 64;
  const int64_t ro = (int64_t)s * (a.pt.nrows + 1);
  const int *irow = (ADJ ? a.pt.rrow : a.pt.srow) + ro, *rrow = a.pt.rrow + ro;
  const int64_t *icell = ADJ ? a.pt.urec_cell : a.pt.usrc_cell;
  const int *iptr = ADJ ? a.pt.urec_ptr : a.pt.usrc_ptr, *ilist = ADJ ? a.pt.urec_list : a.pt.usrc_list;
  const T *tf = ADJ ? a.res + a.pt.off_tr[s] : a.srctf + a.pt.off_tf[s];
  // bounds of the rows' points, one row per lane
  const int jl = min(W.j0 + min(W.lane, R), a.nz);
  const int ib = irow[min(jl, a.nz)], rb = (!ADJ && a.traces) ? rrow[min(jl, a.nz)] : 0;
  W.imask = W.rmask = 0;
#pragma unroll
  for (int r = 0; r < R; r++) {
    if (__shfl(ib, r) != __shfl(ib, r + 1)) W.imask |= 1 << r;
    if (__shfl(rb, r) != __shfl(rb, r + 1)) W.rmask |= 1 << r;
  }
  W.imask = __builtin_amdgcn_readfirstlane(W.imask);
  W.rmask = __builtin_amdgcn_readfirstlane(W.rmask);
  if (!(W.imask | W.rmask)) return;
  for (int r = 0; r < R; r++) {
    const int64_t c0 = (int64_t)(W.j0 + r) * a.nx + X0;
    if (W.imask >> r & 1) {
      L.inj[W.w * R + r][W.lane] = 0;
      __builtin_amdgcn_wave_barrier();
      const int q1 = __shfl(ib, r + 1);
      for (int q = __shfl(ib, r) + W.lane; q < q1; q += TX) {
        const int64_t o = icell[q] - c0;
        if (o < 0 || o >= TX) continue;
        const int k0 = iptr[q], cnt = iptr[q + 1] - k0;
        const int slot = cnt <= SN_SLOTS ? atomicAdd(&L.used, cnt) : SN_SLOTS;
        if (slot + cnt > SN_SLOTS) {
          L.inj[W.w * R + r][o] = -1;
          continue;
        }
        for (int k = 0; k < cnt; k++) {
          const T *v = tf + (int64_t)nts * ilist[k0 + k] + (la - 1);
          for (int m = 0; m < nl; m++) L.val[m][slot + k] = v[ADJ ? -m : m];
        }
        L.inj[W.w * R + r][o] = (short)((slot + 1) | cnt << 7);
      }
    }
    if (W.rmask >> r & 1) {
      L.rec[W.w * R + r][W.lane] = 0;
      __builtin_amdgcn_wave_barrier();
      const int q1 = __shfl(rb, r + 1);
      for (int q = __shfl(rb, r) + W.lane; q < q1; q += TX) {
        const int64_t o = a.pt.urec_cell[q] - c0;
        if (o < 0 || o >= TX) continue;
        const int k0 = a.pt.urec_ptr[q], cnt = a.pt.urec_ptr[q + 1] - k0;
        const int first = cnt <= 127 ? atomicAdd(&L.rused, cnt) : SN_RECS;
        if (first + cnt > SN_RECS) {
          L.rec[W.w * R + r][o] = -1;
          continue;
        }
        for (int k = 0; k < cnt; k++) L.col[first + k] = a.pt.urec_list[k0 + k];
        L.rec[W.w * R + r][o] = (short)((first + 1) | cnt << 8);
      }
    }
  }
}

}  // namespace swx
