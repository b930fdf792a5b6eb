"""1D time loops with the fields in registers against the general loops
(SWX_1D_RESIDENT=0), which the oracle tests pin: seismograms, misfit and
gradient bitwise equal at the sizes where the workgroup's shape changes, with
shots of uneven length, several points on a cell, points on the outermost
cells, more receivers than threads, and too many to stage (both general)."""
import numpy as np
import pytest

import seismicwaves as sw

pytestmark = pytest.mark.gpu


def _run(monkeypatch, resident, vd, dtype, nx, halo, nts, nrec, cf, seed):
    monkeypatch.setenv("SWX_1D_RESIDENT", "1" if resident else "0")
    rng = np.random.default_rng(seed)
    h, dt = 5.0, 5e-4
    vp = rng.uniform(1500.0, 4000.0, nx).astype(dtype)
    shots, misfits = [], []
    for nt in nts:
        cells = rng.integers(0, nx, (3, 1)).astype(float)
        cells[1] = cells[0]                       # two sources on one cell
        cells[2] = 0                              # and one on the edge
        tf = rng.standard_normal((nt, 3)).astype(dtype)
        rec = np.concatenate([rng.integers(0, nx, nrec - 2), [0, nx - 1]])[:, None].astype(float)
        shots.append(sw.ScalarShot(sw.ScalarSources(cells * h, tf, float(rng.uniform(8.0, 15.0))),
                                   sw.ScalarReceivers(rec * h, nt, dtype=dtype)))
        misfits.append(sw.L2Misfit(rng.standard_normal((nt, nrec)).astype(dtype)))
    mp = (sw.VpRhoAcousticVDMaterialProperties(vp, rng.uniform(1500.0, 2500.0, nx).astype(dtype)) if vd
          else sw.VpAcousticCDMaterialProperties(vp))
    params = sw.InputParametersAcoustic(max(nts), dtype(dt), (nx,), (h,),
                                        sw.CPMLBoundaryConditionParameters(halo=halo, freeboundtop=False))
    g, mis = sw.swgradient(params, mp, shots, misfits, runparams=sw.RunParameters(erroronPPW=False),
                           gradparams=sw.GradParameters(check_freq=cf, compute_misfit=True))
    return g, mis, [s.recs.seismograms for s in shots]


@pytest.mark.parametrize("vd", [False, True])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("nx,halo,nrec", [(45, 20, 3), (256, 0, 300), (257, 1, 9), (1024, 20, 5), (1025, 30, 5),
                                          (2049, 20, 40), (4096, 64, 200), (4097, 20, 5), (300, 65, 5),
                                          (300, 10, 600)])
def test_resident_equals_general(monkeypatch, vd, dtype, nx, halo, nrec):
    if nx < 2 * halo + 3:
        pytest.skip("grid smaller than its C-PML")
    for nts, cf in (([131, 90, 64], 50), ([73], 9)):
        print(f"[1d {'vd' if vd else 'cd'} {np.dtype(dtype).name} nx {nx} halo {halo} nrec {nrec} nt {nts}]", flush=True)
        args = (vd, dtype, nx, halo, nts, nrec, cf, 7 + nx)
        ga, ma, sa = _run(monkeypatch, True, *args)
        gb, mb, sb = _run(monkeypatch, False, *args)
        assert ma == mb
        for a, b in zip(sa, sb):
            assert np.max(np.abs(b)) > 0 and np.array_equal(a, b)
        for key in gb:
            assert np.max(np.abs(gb[key])) > 0 and np.array_equal(ga[key], gb[key]), key
