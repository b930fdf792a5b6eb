// Points of a block that steps a 64-column window of registers by several
// levels per launch: the injected values of all its levels and the trace of
// every recorded cell, staged once in LDS.
#pragma once
#include "swx_device.hpp"

namespace swx {

constexpr int SN_MAX = 8;        // most levels per launch
constexpr int SN_SLOTS = 126;    // staged point values per level
constexpr int SN_RECS = 254;     // receivers on cells with several of them whose traces are kept

// H rows of 64 columns.  A cell with one point is the rule: its trace, or where
// no slot is left the column of its values, stands in the cell's entry itself:
// a search per cell and level made windows full of points slower than one-level
// launches.  500 x 400, 4 shots, float32, forward of 100 levels, with 16 full
// rows of receivers: CD 2.05 -> 0.47 ms (one level per launch 1.18), VD 2.09 ->
// 0.93 (2.1); with one full row CD 0.43 -> 0.39.
// ~(2 x) and ~(2 x + 1) are negative numbers for two kinds of x >= 0.
template <typename T, int H>
struct LevelPoints {
  int inj[H][64];              // staged values of a cell's points: slot + 1 and, above bit 7, their number;
                               // 0: no point; ~(2 u): points of unique cell u, ~(2 c + 1): one, column c
  int rec[H][64];              // trace + 1 of a cell's receiver; 0: none; ~(2 u): receivers of unique cell u,
                               // ~(2 x + 1): x = first entry of col and, above bit 8, their number
  T val[SN_MAX][SN_SLOTS];
  int col[SN_RECS];            // traces of the window's receivers on cells with several
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
  const T *tf = (ADJ ? a.res + a.pt.off_tr[s] : a.srctf + a.pt.off_tf[s]) + (l - 1);
  const int x = ~e >> 1;
  if (~e & 1) {
    add(tf[(int64_t)nts * x]);
    return;
  }
  const int *ptr = ADJ ? a.pt.urec_ptr : a.pt.usrc_ptr, *list = ADJ ? a.pt.urec_list : a.pt.usrc_list;
#pragma clang loop unroll(disable)
  for (int k = ptr[x]; k < ptr[x + 1]; k++) add(tf[(int64_t)nts * list[k]]);
}

// Records p at the receivers of the lane's cell of row r; tr: trace 0 of the
// shot at the level.
template <typename T, int R, typename Args, typename Lds>
__device__ __forceinline__ void level_record(const Args &a, const Lds &L, const LevelWin &W, int nts, int r, T *tr,
                                             T p) {
  const int e = L.rec[W.w * R + r][W.lane];
  if (e > 0) {
    tr[(int64_t)nts * (e - 1)] = p;
  } else if (e < 0) {
    const int x = ~e >> 1;
    if (~e & 1) {
#pragma clang loop unroll(disable)
      for (int k = 0; k < x >> 8; k++) tr[(int64_t)nts * L.col[(x & 255) + k]] = p;
    } else {
#pragma clang loop unroll(disable)
      for (int k = a.pt.urec_ptr[x]; k < a.pt.urec_ptr[x + 1]; k++) tr[(int64_t)nts * a.pt.urec_list[k]] = p;
    }
  }
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
  // The unique cells of the rows in the window: lane r finds the first one of
  // row r, lane 32 + r the end, all in one search.
  static_assert(R <= 32, "one lane per row and bound");
  auto bounds = [&](const int *row, const int64_t *cell) {
    const int r = W.lane & 31, j = W.j0 + r;
    int lo = 0, hi = 0;
    if (r < R && j < a.nz) {
      lo = row[j];
      hi = row[j + 1];
    }
    const int64_t c = (int64_t)j * a.nx + X0 + (W.lane & 32 ? TX : 0);
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (cell[mid] < c) lo = mid + 1;
      else hi = mid;
    }
    return lo;
  };
  const int ib = bounds(irow, icell), rb = !ADJ && a.traces ? bounds(rrow, a.pt.urec_cell) : 0;
  const int ie = __shfl_down(ib, 32), re = __shfl_down(rb, 32);
  W.imask = (int)__ballot(W.lane < R && ib != ie);
  W.rmask = (int)__ballot(W.lane < R && rb != re);
  if (!(W.imask | W.rmask)) return;
  for (int r = 0; r < R; r++) {
    const int64_t c0 = (int64_t)(W.j0 + r) * a.nx + X0;
    if (W.imask >> r & 1) {
      L.inj[W.w * R + r][W.lane] = 0;
      __builtin_amdgcn_wave_barrier();
      const int q = __shfl(ib, r) + W.lane;
      if (q < __shfl(ie, r)) {
        const int o = (int)(icell[q] - c0);
        const int k0 = iptr[q], cnt = iptr[q + 1] - k0;
        const int slot = cnt <= SN_SLOTS ? atomicAdd(&L.used, cnt) : SN_SLOTS;
        if (slot + cnt > SN_SLOTS) {
          L.inj[W.w * R + r][o] = cnt == 1 ? ~(2 * ilist[k0] + 1) : ~(2 * q);
        } else {
          for (int k = 0; k < cnt; k++) {
            const T *v = tf + (int64_t)nts * ilist[k0 + k] + (la - 1);
            for (int m = 0; m < nl; m++) L.val[m][slot + k] = v[ADJ ? -m : m];
          }
          L.inj[W.w * R + r][o] = (slot + 1) | cnt << 7;
        }
      }
    }
    if (W.rmask >> r & 1) {
      L.rec[W.w * R + r][W.lane] = 0;
      __builtin_amdgcn_wave_barrier();
      const int q = __shfl(rb, r) + W.lane;
      if (q < __shfl(re, r)) {
        const int o = (int)(a.pt.urec_cell[q] - c0);
        const int k0 = a.pt.urec_ptr[q], cnt = a.pt.urec_ptr[q + 1] - k0;
        const int first = cnt > 1 && cnt <= SN_RECS ? atomicAdd(&L.rused, cnt) : SN_RECS;
        int e = ~(2 * q);
        if (cnt == 1) {
          e = a.pt.urec_list[k0] + 1;
        } else if (first + cnt <= SN_RECS) {
          for (int k = 0; k < cnt; k++) L.col[first + k] = a.pt.urec_list[k0 + k];
          e = ~(2 * (first | cnt << 8) + 1);
        }
        L.rec[W.w * R + r][o] = e;
      }
    }
  }
}

}  // namespace swx
