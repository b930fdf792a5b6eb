"""VD 2D tile codes that take the shots in groups (code + 1000 k: 2^k shots),
chosen for the first batch of a call, on a later batch that the group does not
divide: seismograms and per-shot gradients bitwise those of one shot per batch."""
import numpy as np
import pytest

import seismicwaves as sw

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fwd,adj", [(1316, 1316), (2308, 2316), (2016, 1016)])
@pytest.mark.parametrize("nshots", [5, 6, 7])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_group_that_does_not_divide_the_batch(monkeypatch, dtype, nshots, fwd, adj):
    n, h, dt, nt, nrec = (140, 75), 5.0, 5e-4, 31, 12
    rng = np.random.default_rng(nshots)
    mp = sw.VpRhoAcousticVDMaterialProperties(rng.uniform(1500.0, 4000.0, n).astype(dtype),
                                              rng.uniform(1800.0, 2400.0, n).astype(dtype))
    params = sw.InputParametersAcoustic(nt, dtype(dt), n, (h, h),
                                        sw.CPMLBoundaryConditionParameters(halo=10, freeboundtop=False))
    shots, misfits = [], []
    for k in range(nshots):
        src, rec = (np.stack([rng.integers(0, m, c) for m in n], 1) * h for c in (2, nrec))
        shots.append(sw.ScalarShot(sw.ScalarSources(src, rng.standard_normal((nt, 2)).astype(dtype), 9.0 + k),
                                   sw.ScalarReceivers(rec, nt, dtype=dtype)))
        misfits.append(sw.L2Misfit(rng.standard_normal((nt, nrec)).astype(dtype)))
    monkeypatch.setenv("SWX_VD2D_TILE_FWD", str(fwd))
    monkeypatch.setenv("SWX_VD2D_TILE_ADJ", str(adj))

    def run(batch):
        print(f"[vd2d groups {fwd} {adj} {np.dtype(dtype).name} {nshots} shots, {batch} per batch]", flush=True)
        ws = sw.build_wavesim(params, mp, runparams=sw.RunParameters(erroronPPW=False, max_batch=batch),
                              gradparams=sw.GradParameters(check_freq=9), gradient=True)
        g = sw.swgradient(ws, mp, shots, misfits, per_shot_gradients=True)
        return g, [s.recs.seismograms.copy() for s in shots], list(ws._plan.info().kernel_variant)

    (ref, refs, _), (g, seis, variant) = run(1), run(4)
    assert all(np.max(np.abs(v)) > 0 for r in ref for v in r.values())
    assert all(np.array_equal(a, b) for a, b in zip(refs, seis))
    assert all(np.array_equal(a[key], b[key]) for a, b in zip(ref, g) for key in a)
    # the codes of the last batch, of 1, 2 or 3 shots
    assert variant == [c if (nshots - 4) % (1 << c // 1000) == 0 else c % 1000 for c in (fwd, adj)]
