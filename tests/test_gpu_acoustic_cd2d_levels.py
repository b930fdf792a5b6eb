"""Several CD 2D levels per launch (cd2d_stepn_kernel) against one-level
launches (SWX_CD2D_STEPS=1, pinned by the oracle tests): seismograms,
snapshots, misfit and gradient bitwise equal for every window shape and
several numbers of levels, on grids of one and of many windows, with shots of
uneven length, points on window borders and edges, several points on a cell,
and more points in a window than are staged."""
import numpy as np
import pytest

import seismicwaves as sw

pytestmark = pytest.mark.gpu


def _run(monkeypatch, steps, shape, dtype, n, halo, nts, nrec, cf, seed):
    monkeypatch.setenv("SWX_CD2D_STEPS", str(steps))
    if shape is None:
        monkeypatch.delenv("SWX_CD2D_SHAPE", raising=False)
    else:
        monkeypatch.setenv("SWX_CD2D_SHAPE", str(shape))
    rng = np.random.default_rng(seed)
    h, dt = 5.0, 5e-4
    vp = rng.uniform(1500.0, 4000.0, n).astype(dtype)
    shots, misfits = [], []
    for k, nt in enumerate(nts):
        src = np.stack([rng.integers(0, m, 5) for m in n], 1).astype(float)
        src[1] = src[0]
        src[2] = [min(48 + k, n[0] - 1), min(16, n[1] - 1)]
        rec = np.stack([rng.integers(0, m, nrec) for m in n], 1).astype(float)
        rec[: nrec // 2, 1] = min(17, n[1] - 1)      # a line of receivers
        rec[-1] = [0, n[1] - 1]
        tf = rng.standard_normal((nt, 5)).astype(dtype)
        shots.append(sw.ScalarShot(sw.ScalarSources(src * h, tf, float(rng.uniform(8.0, 15.0))),
                                   sw.ScalarReceivers(rec * h, nt, dtype=dtype)))
        misfits.append(sw.L2Misfit(rng.standard_normal((nt, nrec)).astype(dtype)))
    mp = sw.VpAcousticCDMaterialProperties(vp)
    params = sw.InputParametersAcoustic(max(nts), dtype(dt), n, (h, h),
                                        sw.CPMLBoundaryConditionParameters(halo=halo, freeboundtop=False))
    g, mis = sw.swgradient(params, mp, shots, misfits, runparams=sw.RunParameters(erroronPPW=False),
                           gradparams=sw.GradParameters(check_freq=cf, compute_misfit=True))
    snaps = sw.swforward(params, mp, shots, runparams=sw.RunParameters(erroronPPW=False, snapevery=11))
    return g["vp"], mis, [s.recs.seismograms for s in shots], snaps


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n,halo,nts,nrec", [((64, 32), 8, [40], 9), ((65, 33), 0, [41, 30], 40),
                                             ((150, 140), 20, [37, 26, 34], 700), ((301, 70), 30, [45], 60)])
def test_levels_per_launch_agree_bitwise(monkeypatch, dtype, n, halo, nts, nrec):
    args = (dtype, n, halo, nts, nrec, 13, 5 + n[0])
    ref = _run(monkeypatch, 1, None, *args)
    assert np.max(np.abs(ref[0])) > 0 and all(np.max(np.abs(s)) > 0 for s in ref[2])
    shapes = (20, 11, 22) if dtype == np.float32 else (21, 22)
    for steps, shape in [(8, None)] + [(k, sh) for sh in shapes for k in (2, 5, 8)]:
        print(f"[cd2d levels {steps} shape {shape} {np.dtype(dtype).name} {n} halo {halo} nrec {nrec}]", flush=True)
        g, mis, seis, snaps = _run(monkeypatch, steps, shape, *args)
        assert np.array_equal(g, ref[0]) and mis == ref[1]
        assert all(np.array_equal(a, b) for a, b in zip(seis, ref[2]))
        for a, b in zip(snaps, ref[3]):
            assert sorted(a) == sorted(b)
            assert all(np.array_equal(a[it]["pcur"], b[it]["pcur"]) for it in b)
