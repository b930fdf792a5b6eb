"""Elastic 2D row march (el_row_kernel) against the two-launch steps
(SWX_EL2D_VARIANT_*=1): seismograms and gradients bitwise equal, on grids
narrower than a window, of exactly one and two windows and one column more,
with and without the free surface, halos of zero cells up to strips that fill
the grid, both source kinds with sources next to strips, window borders and
each other, lines of receivers, shots of uneven length, and chunks of one row
up to the largest."""
import numpy as np
import pytest

import seismicwaves as sw

pytestmark = pytest.mark.gpu


def _run(monkeypatch, variant, rows, dtype, kind, n, halo, freetop, nts, nrec, cf, seed, nsrc=2):
    monkeypatch.setenv("SWX_EL2D_VARIANT_FWD", variant)
    monkeypatch.setenv("SWX_EL2D_VARIANT_ADJ", variant)
    if rows is None:
        monkeypatch.delenv("SWX_EL2D_ROWS", raising=False)
        if variant == "3":       # the default rule
            monkeypatch.delenv("SWX_EL2D_VARIANT_FWD")
            monkeypatch.delenv("SWX_EL2D_VARIANT_ADJ")
    else:
        monkeypatch.setenv("SWX_EL2D_ROWS", str(rows))
    rng = np.random.default_rng(seed)
    h, dt = 10.0, 1e-3
    rho = rng.uniform(1900.0, 2300.0, n)
    vp = rng.uniform(2600.0, 3200.0, n)
    mu = rho * (vp / 1.8) ** 2
    mp = sw.ElasticIsoMaterialProperties(*[x.astype(dtype) for x in (rho * vp ** 2 - 2 * mu, mu, rho)])
    lo, hi = np.array([6.0, 6.0]), np.array([n[0] - 8.0, n[1] - 8.0])
    shots, misfits = [], []
    for k, nt in enumerate(nts):
        src = rng.uniform(lo, hi, (nsrc, 2))
        src[1] = src[0] + [1.3, 0.2]
        src[0, 0] = min(57.3 + k, n[0] - 8.0)
        rec = rng.uniform(lo, hi, (nrec, 2))
        rec[: nrec // 2, 1] = rec[0, 1]
        recs = sw.VectorReceivers(rec * h, nt, dtype=dtype)
        if kind == "mt":
            mom = [sw.MomentTensor2D(*rng.uniform(-1e3, 1e3, 3)) for _ in range(nsrc)]
            srcs = sw.MomentTensorSources(src * h, rng.standard_normal((nt, nsrc)).astype(dtype), mom, 6.0)
            shots.append(sw.MomentTensorShot(srcs, recs))
        else:
            srcs = sw.ExternalForceSources(src * h, 1e3 * rng.standard_normal((nt, 2, nsrc)).astype(dtype), 6.0)
            shots.append(sw.ExternalForceShot(srcs, recs))
        misfits.append(sw.L2Misfit(rng.standard_normal((nt, 2, nrec)).astype(dtype)))
    params = sw.InputParametersElastic(max(nts), dt, n, (h, h),
                                       sw.CPMLBoundaryConditionParameters(halo=halo, rcoef=1e-4, freeboundtop=freetop))
    ws = sw.build_wavesim(params, mp, runparams=sw.RunParameters(erroronPPW=False),
                          gradparams=sw.GradParameters(check_freq=cf, compute_misfit=True), gradient=True)
    g, mis = sw.run_swgradient(ws, mp, shots, misfits)
    # moment tensors of many sources in one tile keep the former steps
    if variant != "3" or (kind == "ef" or nsrc == 2):
        assert list(ws._plan.info().kernel_variant) == [int(variant)] * 2
    return g, mis, [s.recs.seismograms.copy() for s in shots]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("kind,n,halo,freetop,nts,nrec", [("mt", (40, 33), 0, True, [30], 5),
                                                          ("ef", (40, 37), 0, False, [30, 22], 5),
                                                          ("mt", (64, 61), 10, False, [40, 31], 9),
                                                          ("ef", (65, 45), 12, True, [37], 30),
                                                          ("mt", (122, 70), 20, True, [33, 41, 28], 60),
                                                          ("ef", (123, 150), 15, True, [35, 26], 40),
                                                          ("mt", (301, 96), 5, False, [31], 20)])
def test_row_march_agrees_bitwise(monkeypatch, dtype, kind, n, halo, freetop, nts, nrec):
    args = (dtype, kind, n, halo, freetop, nts, nrec, 11, 7 + n[0])
    ref = _run(monkeypatch, "1", None, *args)
    assert all(np.max(np.abs(ref[0][k])) > 0 for k in ref[0]) and all(np.max(np.abs(s)) > 0 for s in ref[2])
    for rows in (None, 1, 2, 5, 13, 56):
        print(f"[el2d rows {rows} {kind} {np.dtype(dtype).name} {n} halo {halo} freetop {freetop}]", flush=True)
        g, mis, seis = _run(monkeypatch, "3", rows, *args)
        assert mis == ref[1]
        assert all(np.array_equal(a, b) for a, b in zip(seis, ref[2]))
        for k in ref[0]:
            assert np.array_equal(g[k], ref[0][k]), k


@pytest.mark.parametrize("kind", ["mt", "ef"])
def test_more_source_taps_than_a_wave_lists(monkeypatch, kind):
    args = (np.float32, kind, (150, 90), 10, False, [25, 31], 20, 11, 3, 12)
    ref = _run(monkeypatch, "1", None, *args)
    print(f"[el2d rows, 12 sources, {kind}]", flush=True)
    g, mis, seis = _run(monkeypatch, "3", 40, *args)
    assert mis == ref[1] and all(np.array_equal(a, b) for a, b in zip(seis, ref[2]))
    assert all(np.array_equal(g[k], ref[0][k]) for k in ref[0])
