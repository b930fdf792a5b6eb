"""Launch shapes are timed once per plan: a second call on a wave simulation
whose batches differ in size or points times none (the library says on stderr,
with SWX_PROGRESS set, when it does)."""
import os
import subprocess
import sys

import pytest

from conftest import PKG_ROOT

pytestmark = pytest.mark.gpu

VD2D = """
n, nt, nshots, batch = (600, 500), 4, 12, 11      # 11 shots: single steps, 1 shot: several levels
mp = sw.VpRhoAcousticVDMaterialProperties(np.full(n, 2000.0), np.full(n, 2000.0))
options = {}
at = np.array([[1500.0, 1200.0]])
shots = [sw.ScalarShot(sw.ScalarSources(at, np.ones((nt, 1)), 9.0), sw.ScalarReceivers(at, nt))
         for _ in range(nshots)]
misfits = [sw.L2Misfit(np.zeros((nt, 1))) for _ in shots]
params = sw.InputParametersAcoustic(nt, 5e-4, n, (5.0, 5.0), sw.CPMLBoundaryConditionParameters(halo=10))
"""

ELASTIC = """
n, nt, batch = (90, 80), 4, 1      # the second shot's moment tensor reaches a stress cell that no step updates
rho = np.full(n, 2000.0)
mp = sw.ElasticIsoMaterialProperties(rho * 2000.0 ** 2, rho * 1500.0 ** 2, rho)
rec = np.array([[250.0, 200.0]])
shots = [sw.MomentTensorShot(sw.MomentTensorSources(np.array([at]), np.ones((nt, 1)),
                                                    [sw.MomentTensor2D(1e6, 1e6, 0.0)], 9.0),
                             sw.VectorReceivers(rec, nt)) for at in ([200.0, 200.0], [0.0, 200.0])]
misfits = [sw.L2Misfit(np.zeros((nt, 2, 1))) for _ in shots]
params = sw.InputParametersElastic(nt, 5e-4, n, (5.0, 5.0), sw.CPMLBoundaryConditionParameters(halo=10))
options = {"sincinterp": False}
"""

RUN = """
import sys
sys.path.insert(0, sys.argv[1])
import numpy as np
import seismicwaves as sw
{problem}
ws = sw.build_wavesim(params, mp, runparams=sw.RunParameters(erroronPPW=False, max_batch=batch), gradient=True,
                      gradparams=sw.GradParameters(check_freq=2), **options)
for call in (1, 2, 3):
    print("call", call, file=sys.stderr, flush=True)
    sw.swgradient(ws, mp, shots, misfits)
"""


@pytest.mark.parametrize("problem", [VD2D, ELASTIC], ids=["vd2d", "elastic"])
def test_second_call_times_no_launch_shape(problem):
    env = {k: v for k, v in os.environ.items() if not k.startswith("SWX_") or k == "SWX_LIBRARY"}
    r = subprocess.run([sys.executable, "-c", RUN.replace("{problem}", problem), PKG_ROOT], stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT, text=True, timeout=100, env={**env, "SWX_PROGRESS": "1"})
    assert r.returncode == 0, r.stdout[-2000:]
    first, second, third = r.stdout.split("call ")[1:]
    assert "launch shapes timed" in first
    assert "launch shapes timed" not in second and "launch shapes timed" not in third
