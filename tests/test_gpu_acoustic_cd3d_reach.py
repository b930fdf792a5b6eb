"""A pinned CD 3D row march (SWX_CD3D_VARIANT=301) is refused where its 32-bit
byte offsets do not reach over a shot's field, before any field is allocated;
the field just below takes it."""
import numpy as np
import pytest

from seismicwaves import _native

pytestmark = pytest.mark.gpu


def _plan(dtype, n):
    return _native.Plan(physics=_native.SWX_ACOUSTIC_CD, dtype=dtype, n=n, h=(5.0, 5.0, 5.0), dt=4e-4, halo=2,
                        freetop=False, max_shots=1, nt_max=4, check_freq=1, gradient=False)


@pytest.mark.parametrize("dtype,n", [(np.float32, (1024, 1024, 1024)), (np.float64, (1024, 1024, 512))])
def test_pinned_row_march_is_refused_from_4_gib_on(monkeypatch, dtype, n):
    monkeypatch.setenv("SWX_CD3D_VARIANT", "301")
    with pytest.raises(AssertionError, match="below 4 GiB"):
        _plan(dtype, n)
    _plan(dtype, (n[0], n[1], n[2] - 1)).close()
    monkeypatch.setenv("SWX_CD3D_VARIANT", "4")
    _plan(dtype, n).close()
