"""CD 3D row march with the longest chunks, on grids deep enough that the
planes loaded ahead of a chunk lie outside both z strips: bitwise equal to the
tile kernel, and the chunk that ran is the one reported."""
import numpy as np
import pytest

import seismicwaves as sw
from test_gpu_acoustic_cd3d_rows import _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n,halo", [((40, 24, 140), 10), ((66, 9, 131), 2)])
def test_long_chunks_agree_bitwise(monkeypatch, dtype, n, halo):
    args = (dtype, n, halo, [22, 17], 30, 9, 5)
    ref = _run(monkeypatch, 4, 24, *args)
    for chunk in (61, 62, 63, 64, 100):
        print(f"[cd3d chunk {chunk} {np.dtype(dtype).name} {n} halo {halo}]", flush=True)
        g, mis, seis, _ = _run(monkeypatch, 301, chunk, *args)
        assert np.max(np.abs(g)) > 0 and np.array_equal(g, ref[0]) and mis == ref[1]
        assert all(np.array_equal(a, b) for a, b in zip(seis, ref[2]))


@pytest.mark.parametrize("variant,chunk,used", [(301, 100, 62), (301, 62, 62), (301, 9, 9), (4, 100, 100)])
def test_reported_chunk_is_the_one_used(monkeypatch, variant, chunk, used):
    monkeypatch.setenv("SWX_CD3D_VARIANT", str(variant))
    monkeypatch.setenv("SWX_CD3D_ZCHUNK", str(chunk))
    n, h, nt = (20, 12, 70), 5.0, 4
    params = sw.InputParametersAcoustic(nt, 4e-4, n, (h, h, h),
                                        sw.CPMLBoundaryConditionParameters(halo=3, freeboundtop=False))
    mp = sw.VpAcousticCDMaterialProperties(np.full(n, 2000.0))
    ws = sw.build_wavesim(params, mp, runparams=sw.RunParameters(erroronPPW=False), gradient=False)
    at = np.array([[10 * h, 6 * h, 30 * h]])
    shot = sw.ScalarShot(sw.ScalarSources(at, np.ones((nt, 1)), 10.0), sw.ScalarReceivers(at, nt))
    sw.swforward(ws, mp, [shot])
    assert list(ws._plan.info().kernel_variant) == [variant, used]
