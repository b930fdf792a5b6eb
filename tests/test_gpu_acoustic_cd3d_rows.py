"""CD 3D row march (cd3d_row_kernel) against the tile kernel without its LDS
stage and lean tiles (SWX_CD3D_VARIANT=4, SWX_CD3D_LEAN=0): seismograms,
snapshots, misfit and gradient bitwise equal, on grids narrower than a window,
of exactly one and two windows and one more, with odd numbers of rows, strips
that fill the grid and none, shots of uneven length, points on window borders
and edges and several on a cell, and chunks of one plane up to more than the
grid has."""
import numpy as np
import pytest

import seismicwaves as sw

pytestmark = pytest.mark.gpu


def _run(monkeypatch, variant, chunk, dtype, n, halo, nts, nrec, cf, seed):
    for name, value in (("SWX_CD3D_VARIANT", variant), ("SWX_CD3D_ZCHUNK", chunk)):
        if value is None:
            monkeypatch.delenv(name, raising=False)
        else:
            monkeypatch.setenv(name, str(value))
    monkeypatch.setenv("SWX_CD3D_LEAN", "0" if variant == 4 else "1")
    rng = np.random.default_rng(seed)
    h, dt = 5.0, 4e-4
    vp = rng.uniform(1500.0, 4000.0, n).astype(dtype)
    shots, misfits = [], []
    for k, nt in enumerate(nts):
        src = np.stack([rng.integers(0, m, 6) for m in n], 1).astype(float)
        src[1] = src[0]
        src[2, 0] = min(61 + k, n[0] - 1)
        rec = np.stack([rng.integers(0, m, nrec) for m in n], 1).astype(float)
        rec[: nrec // 2, 1:] = rec[0, 1:]            # a line of receivers
        rec[-1] = [n[0] - 1, 0, n[2] - 1]
        tf = rng.standard_normal((nt, 6)).astype(dtype)
        shots.append(sw.ScalarShot(sw.ScalarSources(src * h, tf, float(rng.uniform(8.0, 15.0))),
                                   sw.ScalarReceivers(rec * h, nt, dtype=dtype)))
        misfits.append(sw.L2Misfit(rng.standard_normal((nt, nrec)).astype(dtype)))
    mp = sw.VpAcousticCDMaterialProperties(vp)
    params = sw.InputParametersAcoustic(max(nts), dtype(dt), n, (h, h, h),
                                        sw.CPMLBoundaryConditionParameters(halo=halo, freeboundtop=False))
    g, mis = sw.swgradient(params, mp, shots, misfits, runparams=sw.RunParameters(erroronPPW=False),
                           gradparams=sw.GradParameters(check_freq=cf, compute_misfit=True))
    snaps = sw.swforward(params, mp, shots, runparams=sw.RunParameters(erroronPPW=False, snapevery=7))
    return g["vp"], mis, [s.recs.seismograms for s in shots], snaps


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n,halo,nts,nrec", [((9, 5, 7), 0, [20], 9), ((62, 9, 12), 3, [30, 21], 40),
                                             ((64, 13, 70), 5, [24], 20), ((65, 30, 23), 10, [31, 17, 26], 300),
                                             ((124, 7, 66), 0, [25], 30), ((127, 33, 25), 6, [22, 27], 60)])
def test_row_march_agrees_bitwise(monkeypatch, dtype, n, halo, nts, nrec):
    args = (dtype, n, halo, nts, nrec, 9, 3 + n[0])
    ref = _run(monkeypatch, 4, 24, *args)
    assert np.max(np.abs(ref[0])) > 0 and all(np.max(np.abs(s)) > 0 for s in ref[2])
    for variant, chunk in [(None, None), (301, 1), (301, 2), (301, 5), (301, 64), (301, 100)]:
        print(f"[cd3d rows chunk {chunk} {np.dtype(dtype).name} {n} halo {halo} nrec {nrec}]", flush=True)
        g, mis, seis, snaps = _run(monkeypatch, variant, chunk, *args)
        assert np.array_equal(g, ref[0]) and mis == ref[1]
        assert all(np.array_equal(a, b) for a, b in zip(seis, ref[2]))
        for a, b in zip(snaps, ref[3]):
            assert sorted(a) == sorted(b)
            assert all(np.array_equal(a[it]["pcur"], b[it]["pcur"]) for it in b)
