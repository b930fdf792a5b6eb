"""Moment tensors in the elastic row march: one source, several on a cell (and
more than a wave's width of them), and sources side by side, bitwise equal to
the two-launch steps; and the waves that hold a source do not make a replayed
step slower than those steps."""
import numpy as np
import pytest

import seismicwaves as sw

pytestmark = pytest.mark.gpu


def _problem(dtype, n, at, nt, sinc):
    rng = np.random.default_rng(len(at))
    h = 10.0
    rho = rng.uniform(1900.0, 2300.0, n)
    vp = rng.uniform(2600.0, 3200.0, n)
    mu = rho * (vp / 1.8) ** 2
    mp = sw.ElasticIsoMaterialProperties(*[x.astype(dtype) for x in (rho * vp ** 2 - 2 * mu, mu, rho)])
    mom = [sw.MomentTensor2D(*rng.uniform(-1e3, 1e3, 3)) for _ in at]
    rec = rng.uniform(25.0, np.array(n) - 25.0, (20, 2)) * h
    shot = sw.MomentTensorShot(sw.MomentTensorSources(np.array(at) * h, rng.standard_normal((nt, len(at))).astype(dtype),
                                                      mom, 6.0), sw.VectorReceivers(rec, nt, dtype=dtype))
    params = sw.InputParametersElastic(nt, 1e-3, n, (h, h), sw.CPMLBoundaryConditionParameters(halo=20))
    ws = sw.build_wavesim(params, mp, runparams=sw.RunParameters(erroronPPW=False), gradient=True, sincinterp=sinc,
                          gradparams=sw.GradParameters(check_freq=20))
    return ws, mp, [shot], [sw.L2Misfit(rng.standard_normal((nt, 2, 20)).astype(dtype))]


def _pin(monkeypatch, variant):
    for name in ("SWX_EL2D_VARIANT_FWD", "SWX_EL2D_VARIANT_ADJ"):
        if variant is None:
            monkeypatch.delenv(name, raising=False)
        else:
            monkeypatch.setenv(name, str(variant))


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("at,sinc", [([(60.3, 40.7)], True), ([(57.0, 30.4)], True), ([(50, 40)] * 100, False),
                                     ([(50 + k % 9, 30 + k // 9) for k in range(81)], False),
                                     ([(70, 33), (70, 33), (71, 33), (28, 33)], False)])
def test_moment_tensor_taps_agree_bitwise(monkeypatch, dtype, at, sinc):
    out = []
    for variant in (1, None):
        _pin(monkeypatch, variant)
        ws, mp, shots, misfits = _problem(dtype, (130, 90), at, 45, sinc)
        g = sw.swgradient(ws, mp, shots, misfits)
        assert list(ws._plan.info().kernel_variant) == ([1, 1] if variant else [3, 3])
        out.append((g, shots[0].recs.seismograms.copy()))
    assert np.max(np.abs(out[0][1])) > 0
    assert np.array_equal(out[0][1], out[1][1]) and all(np.array_equal(out[0][0][k], out[1][0][k]) for k in out[0][0])


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("at", [[(180.3, 140.6)], [(180.3, 140.6), (182.3, 141.6)]], ids=["one", "two"])
def test_source_waves_do_not_hold_up_a_step(monkeypatch, dtype, at):
    """Replay and adjoint of 60 steps, best of 8 calls: at most 1.25 times the
    two-launch steps (1.4 to 2 when the source's waves walk along its taps)."""
    best = {1: np.inf, None: np.inf}
    sims = {}
    for variant in best:
        _pin(monkeypatch, variant)
        sims[variant] = _problem(dtype, (400, 300), at, 60, True)
        sw.swgradient(*sims[variant])
    for _ in range(8):
        for variant, args in sims.items():
            _pin(monkeypatch, variant)
            sw.swgradient(*args)
            best[variant] = min(best[variant], args[0]._plan.info().ms_adjoint)
    print(f"[elastic adjoint {np.dtype(dtype).name}] two launches {best[1]:.2f} ms, row march {best[None]:.2f} ms",
          flush=True)
    assert best[None] <= 1.25 * best[1]
