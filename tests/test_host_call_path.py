"""Host side of a call: the spreading of many points against one coordinate
at a time (coeffsinc1d), the position checks against a scalar restatement,
and the velocity range that follows the model last set."""
import logging

import numpy as np
import pytest

import seismicwaves as sw
from seismicwaves.points import coeffsinc1d


@pytest.mark.parametrize("mirror", [False, True])
@pytest.mark.parametrize("shift", [(0.0, 0.0), (2.5, 0.0), (0.0, 3.5), (2.5, 3.5)])
def test_spread_positions_equals_coordinatewise(shift, mirror):
    n, h = (40, 23), (5.0, 7.0)
    rng = np.random.default_rng(4)
    cells = np.stack([rng.integers(0, m, 20) for m in n], 1)
    pos = np.concatenate([cells * h, (np.minimum(cells, np.array(n) - 2) + 0.5) * h,
                          rng.uniform(0, [(m - 1) * d for m, d in zip(n, h)], (30, 2)),
                          [[0.0, 0.0], [(n[0] - 1) * h[0], (n[1] - 1) * h[1]]]])
    got = sw.spread_positions(pos, h, n, shift, mirror)
    assert len(got) == len(pos)
    for p, (ij, w) in zip(pos, got):
        per = [coeffsinc1d(p[d], h[d], n[d], xstart=shift[d], mirror=mirror, xbl=0.0, xbr=(n[d] - 1) * h[d])
               for d in range(2)]
        want = [(i, j) for j in per[1][0] for i in per[0][0]]
        assert np.array_equal(ij, want)
        assert np.array_equal(w, [a * b for b in per[1][1] for a in per[0][1]])


def _sim(dtype, freetop):
    params = sw.InputParametersAcoustic(10, dtype(1e-3), (50, 40), (7.3, 5.1),
                                        sw.CPMLBoundaryConditionParameters(halo=8, freeboundtop=freetop))
    mp = sw.VpAcousticCDMaterialProperties(np.full((50, 40), 2000.0, dtype))
    return sw.build_wavesim(params, mp, runparams=sw.RunParameters(logger=logging.getLogger("positions")))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("freetop", [False, True])
def test_position_checks_equal_scalar_ones(caplog, dtype, freetop):
    ws = _sim(dtype, freetop)
    ext = [(n - 1) * h for n, h in zip(ws.gridsize, ws.spacing)]
    edges = [h * 8 for h in ws.spacing]
    vals = [[dtype(v) for v in (0.0, e / 2, b, np.nextafter(dtype(b), dtype(0)), x - b, x,
                                np.nextafter(dtype(x), dtype(np.inf)), -1e-3)] for x, b in zip(ext, edges)
            for e in (x,)]
    for a in vals[0]:
        for c in vals[1]:
            p = np.array([a, c], dtype=dtype)
            inside = all(0 <= p[k] <= ext[k] for k in range(2))
            warn = sum(not (edges[k] <= p[k] <= ext[k] - edges[k]) for k in range(2) if not (k == 1 and freetop))
            caplog.clear()
            with caplog.at_level(logging.WARNING, logger="positions"):
                if inside:
                    ws.check_positions(p)
                    assert len(caplog.records) == warn
                else:
                    with pytest.raises(AssertionError):
                        ws.check_positions(p)


def test_velocity_range_follows_the_model():
    ws = _sim(np.float64, True)
    vp = np.full((50, 40), 2000.0)
    ws.set_matprop(sw.VpAcousticCDMaterialProperties(vp))
    assert ws.velocity_range() == (2000.0, 2000.0)
    vp[3, 4] = 1500.0
    vp[5, 6] = 2500.0
    ws.set_matprop(sw.VpAcousticCDMaterialProperties(vp))
    assert ws.velocity_range() == (1500.0, 2500.0)
