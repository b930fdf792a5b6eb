"""VD 2D gradients without a C-PML on grids whose last rows fall anywhere in a
wave's rows, with sources and receivers on the last rows of interior columns:
several levels per launch against one-level launches, bitwise."""
import numpy as np
import pytest

import seismicwaves as sw

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("adj", [502, 503])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_last_row_without_cpml(monkeypatch, dtype, adj):
    h, dt, nt, nx = 5.0, 5e-4, 12, 210

    def run(nz, tile):
        monkeypatch.setenv("SWX_VD2D_TILE_ADJ", str(tile))
        rng = np.random.default_rng(nz)
        n = (nx, nz)
        mp = sw.VpRhoAcousticVDMaterialProperties(rng.uniform(1500.0, 4000.0, n).astype(dtype),
                                                  rng.uniform(1800.0, 2400.0, n).astype(dtype))
        params = sw.InputParametersAcoustic(nt, dtype(dt), n, (h, h),
                                            sw.CPMLBoundaryConditionParameters(halo=0, freeboundtop=False))
        at = np.array([[x * h, (nz - 1 - k % 2) * h] for k, x in enumerate((70, 95, 104, 130))])
        shot = sw.ScalarShot(sw.ScalarSources(at, rng.standard_normal((nt, 4)).astype(dtype), 9.0),
                             sw.ScalarReceivers(at, nt, dtype=dtype))
        ws = sw.build_wavesim(params, mp, runparams=sw.RunParameters(erroronPPW=False), gradient=True,
                              gradparams=sw.GradParameters(check_freq=5))
        g = sw.swgradient(ws, mp, [shot], [sw.L2Misfit(rng.standard_normal((nt, 4)).astype(dtype))])
        assert ws._plan.info().kernel_variant[1] == tile
        ws._plan.close()
        return g

    print(f"[vd2d last row {np.dtype(dtype).name} {adj}]", flush=True)
    for nz in range(60, 110):
        ref, g = run(nz, 316), run(nz, adj)
        assert np.max(np.abs(ref["rho"][:, -2])) > 0
        assert all(np.array_equal(g[k], ref[k]) for k in ref), nz
