"""Wave speeds of single-stage inviscid steps with a CFL time step: formed (and
on the first step refreshed) before the time step, and left there for the
caller.  Against the oracle, after the first step and later ones."""
import numpy as np
import pytest

from flurrypp_amd import cases
from flurrypp_amd._native import PATH_FUSED, PATH_MIXED, PATH_STAGED
from flurrypp_amd.solver import Solver
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu

CASES = {
    "bump2d": lambda dt_type: cases.bump2d(nx=9, ny=5, order=2, dt_type=dt_type, time_type=0, cfl=0.3),
    "vortex2d_roe": lambda dt_type: cases.vortex2d(n=6, order=3, dt_type=dt_type, time_type=0, riemann=1, cfl=0.3),
    "bump2d_fixed": lambda dt_type: cases.bump2d(nx=9, ny=5, order=1, dt_type=0, time_type=0, dt=1e-4),
}
# FP64: the stage tests' bar for wave speeds.  Mixed: U at a point is a sum of 4 products with weights of
# up to 2.5 in all (10 roundings of 6e-8), pressure and speed of sound take some 7 more: 1e-6, and as much
# again for the state that the earlier steps left.
RTOL = {PATH_FUSED: 1e-11, PATH_STAGED: 1e-11, PATH_MIXED: 2e-6}


@pytest.mark.parametrize("path", [PATH_FUSED, PATH_MIXED, PATH_STAGED])
@pytest.mark.parametrize("dt_type", [1, 2])
@pytest.mark.parametrize("name", list(CASES))
def test_wave_speeds(name, dt_type, path):
    setup, U = CASES[name](dt_type)
    s, o = Solver(setup.params, setup=setup), Oracle.from_setup(setup)
    # a state away from the free stream, on which the common flux's speed is another than the point's own
    U = U * (1.0 + 0.02 * np.sin(np.arange(U.size)).reshape(U.shape))
    s.initializeSolution(U)
    o.initializeSolution(U, setup.params.dtType)
    if setup.params.dtType == 0:  # left and boundary points alone are written
        s.put("waveSp", np.zeros(s.nFpts * s.nEles))
        o.put("waveSp", np.zeros(s.nFpts * s.nEles))
    for n in (1, 1, 2):
        s.update(n, path=path)
        o.update(n)
        np.testing.assert_allclose(s.get("waveSp"), o.get("waveSp"), rtol=RTOL[path])
        if setup.params.dtType != 0:
            np.testing.assert_allclose(s.calcDt(False), o.calcDt(False), rtol=RTOL[path])
    s.close()
