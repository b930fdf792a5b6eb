"""Several VD 2D levels per launch (vd2d_stepn_kernel) against one-level
launches (SWX_VD2D_TILE_*=316, pinned by the oracle tests): seismograms,
snapshots, misfit and gradient bitwise equal for several numbers of levels, on
grids of one and of many windows, with shots of uneven length, points on window
borders and edges, several points on a cell, and more points in a window than
are staged."""
import numpy as np
import pytest

import seismicwaves as sw

pytestmark = pytest.mark.gpu


def _run(monkeypatch, tile, dtype, n, halo, nts, nrec, cf, seed):
    for name in ("SWX_VD2D_TILE_FWD", "SWX_VD2D_TILE_ADJ"):      # 51n: forward only
        if tile is None:
            monkeypatch.delenv(name, raising=False)
        else:
            monkeypatch.setenv(name, str(tile))
    rng = np.random.default_rng(seed)
    h, dt = 5.0, 5e-4
    vp = rng.uniform(1500.0, 4000.0, n).astype(dtype)
    rho = rng.uniform(1800.0, 2400.0, n).astype(dtype)
    shots, misfits = [], []
    for k, nt in enumerate(nts):
        src = np.stack([rng.integers(0, m, 5) for m in n], 1).astype(float)
        src[1] = src[0]
        src[2] = [min(40 + k, n[0] - 1), min(12, n[1] - 1)]
        rec = np.stack([rng.integers(0, m, nrec) for m in n], 1).astype(float)
        rec[: nrec // 2, 1] = min(17, n[1] - 1)      # a line of receivers
        rec[-1] = [0, n[1] - 1]
        tf = rng.standard_normal((nt, 5)).astype(dtype)
        shots.append(sw.ScalarShot(sw.ScalarSources(src * h, tf, float(rng.uniform(8.0, 15.0))),
                                   sw.ScalarReceivers(rec * h, nt, dtype=dtype)))
        misfits.append(sw.L2Misfit(rng.standard_normal((nt, nrec)).astype(dtype)))
    mp = sw.VpRhoAcousticVDMaterialProperties(vp, rho)
    params = sw.InputParametersAcoustic(max(nts), dtype(dt), n, (h, h),
                                        sw.CPMLBoundaryConditionParameters(halo=halo, freeboundtop=False))
    g, mis = sw.swgradient(params, mp, shots, misfits, runparams=sw.RunParameters(erroronPPW=False),
                           gradparams=sw.GradParameters(check_freq=cf, compute_misfit=True))
    seis = [s.recs.seismograms.copy() for s in shots]
    snaps = sw.swforward(params, mp, shots, runparams=sw.RunParameters(erroronPPW=False, snapevery=11))
    return g, mis, seis + [s.recs.seismograms.copy() for s in shots], snaps


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n,halo,nts,nrec", [((40, 31), 8, [40], 9), ((64, 33), 0, [41, 30], 40),
                                             ((65, 64), 5, [29, 37], 12), ((150, 140), 20, [37, 26, 34], 700),
                                             ((301, 70), 30, [45], 60)])
def test_levels_per_launch_agree_bitwise(monkeypatch, dtype, n, halo, nts, nrec):
    args = (dtype, n, halo, nts, nrec, 13, 5 + n[0])
    ref = _run(monkeypatch, 316, *args)
    assert all(np.max(np.abs(v)) > 0 for v in ref[0].values()) and all(np.max(np.abs(s)) > 0 for s in ref[2])
    for tile in [None, 501, 502, 503, 505, 511, 512, 515] + ([508, 518] if dtype == np.float32 else []):
        print(f"[vd2d levels {tile} {np.dtype(dtype).name} {n} halo {halo} nrec {nrec}]", flush=True)
        g, mis, seis, snaps = _run(monkeypatch, tile, *args)
        assert mis == ref[1] and all(np.array_equal(g[k], ref[0][k]) for k in ref[0])
        assert all(np.array_equal(a, b) for a, b in zip(seis, ref[2]))
        for a, b in zip(snaps, ref[3]):
            assert sorted(a) == sorted(b)
            assert all(np.array_equal(a[it]["pcur"], b[it]["pcur"]) for it in b)
