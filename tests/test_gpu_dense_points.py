"""Several 2D acoustic levels per launch with more sources and receivers in a
window than are staged (whole rows of them, and more on one cell than a window
has slots): bitwise equal to one-level launches, and faster than those."""
import numpy as np
import pytest

import seismicwaves as sw

pytestmark = pytest.mark.gpu

SINGLE = {"cd": {"SWX_CD2D_STEPS": "1"}, "vd": {"SWX_VD2D_TILE_FWD": "316", "SWX_VD2D_TILE_ADJ": "316"}}


def _pin(monkeypatch, kind, single):
    for name, value in SINGLE[kind].items():
        if single:
            monkeypatch.setenv(name, value)
        else:
            monkeypatch.delenv(name, raising=False)


def _sim(kind, dtype, n, src, rec, nt, halo, nshots=1):
    rng = np.random.default_rng(len(rec))
    h, dt = 5.0, 5e-4
    vp = rng.uniform(1500.0, 4000.0, n).astype(dtype)
    mp = (sw.VpAcousticCDMaterialProperties(vp) if kind == "cd"
          else sw.VpRhoAcousticVDMaterialProperties(vp, rng.uniform(1800.0, 2400.0, n).astype(dtype)))
    shots = [sw.ScalarShot(sw.ScalarSources(np.array(src) * h, rng.standard_normal((nt, len(src))).astype(dtype), 9.0),
                           sw.ScalarReceivers(np.array(rec) * h, nt, dtype=dtype)) for _ in range(nshots)]
    params = sw.InputParametersAcoustic(nt, dtype(dt), n, (h, h),
                                        sw.CPMLBoundaryConditionParameters(halo=halo, freeboundtop=True))
    ws = sw.build_wavesim(params, mp, runparams=sw.RunParameters(erroronPPW=False), gradient=True,
                          gradparams=sw.GradParameters(check_freq=25))
    return ws, mp, shots, [sw.L2Misfit(rng.standard_normal((nt, len(rec))).astype(dtype)) for _ in shots]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("kind", ["cd", "vd"])
@pytest.mark.parametrize("many", ["receivers", "sources", "both"])
def test_windows_full_of_points_agree_bitwise(monkeypatch, kind, dtype, many):
    n, nt = (150, 90), 41
    rows = [(i, j) for j in range(20, 36) for i in range(n[0])]
    pile = [(31, 50)] * 300 + [(90, 50)] * 127 + [(91, 50)] * 3
    edges = [(0, 0), (n[0] - 1, 89), (63, 89), (64, 0), (0, 45)]
    src = rows + pile + edges if many != "receivers" else [(75, 40), (75, 40), (3, 4)]
    rec = rows + pile + edges if many != "sources" else [(75, 41), (20, 5)]
    out = []
    for single in (True, False):
        _pin(monkeypatch, kind, single)
        print(f"[{kind} dense {many} {np.dtype(dtype).name} single {single}]", flush=True)
        ws, mp, shots, misfits = _sim(kind, dtype, n, src, rec, nt, 10)
        g = sw.swgradient(ws, mp, shots, misfits)
        variant = list(ws._plan.info().kernel_variant)
        assert (variant[-1] in (11, 316)) == single, variant
        out.append((g, shots[0].recs.seismograms.copy()))
    assert np.max(np.abs(out[0][1])) > 0
    assert np.array_equal(out[0][1], out[1][1]) and all(np.array_equal(out[0][0][k], out[1][0][k]) for k in out[0][0])


@pytest.mark.parametrize("kind", ["cd", "vd"])
def test_full_rows_of_receivers_are_faster_than_single_levels(monkeypatch, kind):
    """500 x 400, 4 shots, float32, 16 rows of receivers: forward of 100 steps, best of 8
    calls: at most 0.75 times the one-level launches (measured 0.40 and 0.44;
    with a search per cell and level 1.7 and 1.0)."""
    n, nt = (500, 400), 100
    rec = [(i, j) for j in range(5, 21) for i in range(n[0])]
    sims, best = {}, {True: np.inf, False: np.inf}
    for single in best:
        _pin(monkeypatch, kind, single)
        sims[single] = _sim(kind, np.float32, n, [(250, 200)], rec, nt, 20, nshots=4)
        sw.swgradient(*sims[single])
    for _ in range(8):
        for single, args in sims.items():
            _pin(monkeypatch, kind, single)
            sw.swgradient(*args)
            best[single] = min(best[single], args[0]._plan.info().ms_forward)
    print(f"[{kind} 16 rows of receivers] single levels {best[True]:.2f} ms, several {best[False]:.2f} ms", flush=True)
    assert best[False] <= 0.75 * best[True]
