"""Band-limited spreading of off-grid sources and receivers over grid taps.

Reference: src/utils/utils.jl:62-214 (kaiser, modd, coeffsinc1D,
spread_positions) as used by the elastic possrcrec_scaletf
(src/models/elastic/ela_models.jl:6-90).  A point becomes, per dimension, a
Kaiser-windowed sinc over the taps i0-r-1 .. i0+r+1 around its nearest grid
point (weights |c| <= 1e-15 dropped), taps beyond the grid are folded back
across the boundary (with a sign flip when `mirror`), coincident taps are
summed, and the 2D weights are the tensor product of the 1D ones.
"""
from __future__ import annotations

import numpy as np

KAISER_R = 4
KAISER_BETA = 6.31


def coeffsinc1d(x0, dx, nx, r=KAISER_R, beta=KAISER_BETA, xstart=0.0, mirror=False, xbl=0.0, xbr=None):
    """1D taps of a band-limited delta at x0 on the grid xstart + dx*(0..nx-1).
    Returns (1-based indices, weights), indices ascending."""
    if xbr is None:
        xbr = (nx - 1) * dx
    xs = xstart + dx * np.arange(nx)
    i0 = int(np.argmin(np.abs(x0 - xs))) + 1
    idx = np.arange(i0 - r - 1, i0 + r + 2)
    xc = (idx - 1) * dx + xstart
    d = xc - x0
    rr = r * dx
    win = np.where(np.abs(d) <= rr, np.i0(beta * np.sqrt(np.clip(1.0 - (d / rr) ** 2, 0.0, None))) / np.i0(beta), 0.0)
    coe = win * np.sinc(d / dx)
    keep = ~(np.abs(coe) <= 1e-15)
    idx, xc, coe = idx[keep], xc[keep], coe[keep]
    left, right = xc < xbl, xc > xbr
    folded = left | right
    if np.any(folded):
        xm = np.where(left, 2 * xbl - xc, 2 * xbr - xc)
        near = np.argmin(np.abs(xm[:, None] - xs[None, :]), axis=1) + 1
        idx = np.where(folded, near, idx)
        if mirror:
            coe = np.where(folded, -coe, coe)
    uniq, inv = np.unique(idx, return_inverse=True)
    w = np.zeros(len(uniq))
    np.add.at(w, inv, coe)
    return uniq.astype(np.int64), w


def _axis_taps(x, dx, nx, r, beta, xstart, mirror, xbl, xbr):
    """coeffsinc1d of every coordinate of x, with the same arithmetic on all
    of them at once (a gather of hundreds of receivers spends its time in
    the window's Bessel functions otherwise: 0.11 ms a coordinate one by one,
    5 us together).  Coordinates whose taps fold back over a boundary go
    through coeffsinc1d."""
    x = np.asarray(x, dtype=np.float64)
    # nearest grid point, the first of two at the same distance
    i0 = np.clip(np.floor((x - xstart) / dx + 0.5).astype(np.int64), 0, nx - 1)
    cand = np.clip(i0[:, None] + np.arange(-1, 2), 0, nx - 1)
    i0 = cand[np.arange(len(x)), np.argmin(np.abs(x[:, None] - (xstart + dx * cand)), axis=1)] + 1
    idx = i0[:, None] + np.arange(-r - 1, r + 2)
    xc = (idx - 1) * dx + xstart
    d = xc - x[:, None]
    rr = r * dx
    win = np.where(np.abs(d) <= rr, np.i0(beta * np.sqrt(np.clip(1.0 - (d / rr) ** 2, 0.0, None))) / np.i0(beta), 0.0)
    coe = win * np.sinc(d / dx)
    keep = ~(np.abs(coe) <= 1e-15)
    folded = np.any(keep & ((xc < xbl) | (xc > xbr)), axis=1)
    return [coeffsinc1d(x[p], dx, nx, r, beta, xstart, mirror, xbl, xbr) if folded[p]
            else (idx[p][keep[p]], coe[p][keep[p]]) for p in range(len(x))]


def spread_positions(positions, spacing, gridsize, shift=(0.0, 0.0), mirror=False, r=KAISER_R, beta=KAISER_BETA):
    """spread_positions with freesurfposition=:ongridbound: per point, the
    taps (ntaps, 2) 1-based and their weights, first dimension fastest."""
    positions = np.atleast_2d(np.asarray(positions, dtype=np.float64))
    per = []
    for d in range(positions.shape[1]):
        # points often share a coordinate (a line of receivers at one depth)
        x, inv = np.unique(positions[:, d], return_inverse=True)
        taps = _axis_taps(x, spacing[d], gridsize[d], r, beta, shift[d], mirror, 0.0, (gridsize[d] - 1) * spacing[d])
        per.append([taps[k] for k in inv.ravel()])
    out = []
    for (ii, wi), (jj, wj) in zip(per[0], per[1]):
        ij = np.empty((len(ii) * len(jj), 2), dtype=np.int64)
        ij[:, 0] = np.tile(ii, len(jj))
        ij[:, 1] = np.repeat(jj, len(ii))
        out.append((ij, (wj[:, None] * wi).ravel()))
    return out


def nearest_taps(idx):
    """One unit tap per point at its nearest grid point (sincinterp = false)."""
    return [(np.asarray(idx[k:k + 1], dtype=np.int64), np.ones(1)) for k in range(idx.shape[0])]
