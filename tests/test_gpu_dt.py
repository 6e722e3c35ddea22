"""The CFL time step's kernel (lanes of a wave over an element's flux points, several
elements in flight, the minimum through atomics) at its edges: one block, several,
a ragged last one, more elements than the blocks take at once, every lane count.
Against the oracle; twice, since a launch leaves the counters for the next."""
import numpy as np
import pytest

from flurrypp_amd import cases
from flurrypp_amd._native import PATH_FUSED, PATH_MIXED
from flurrypp_amd.solver import Solver
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,n,order", [("vortex2d", 2, 0), ("vortex2d", 7, 3), ("vortex2d", 6, 5), ("vortex2d", 100, 1),
                                          ("vortex3d", 3, 0), ("vortex3d", 3, 1), ("vortex3d", 3, 4),
                                          ("vortex3d", 17, 1)])
def test_dt(kind, n, order):
    setup, U = getattr(cases, kind)(n=n, order=order)
    assert setup.params.dtType == 1
    s, o = Solver(setup.params, setup=setup), Oracle.from_setup(setup)
    s.initializeSolution(U)
    o.initializeSolution(U, 1)
    for path in (PATH_FUSED, PATH_FUSED, PATH_MIXED):
        s.update(2, path=path)
        o.update(2)
        # the bars of the parity tests for the FP64 and the mixed path
        rtol = 1e-12 if path == PATH_FUSED else 1e-6
        np.testing.assert_allclose(s.dt, o.dt, rtol=rtol)
        np.testing.assert_allclose(s.get("ele_dt"), o.get("ele_dt"), rtol=rtol)
    s.close()
