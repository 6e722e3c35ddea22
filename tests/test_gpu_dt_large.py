"""The CFL time step's kernel on meshes that take its large blocks (more than 128
or 256 blocks of 256 threads): just past the limit, ragged, with one block's worth over,
and merged meshes, which never do.  Against the oracle; twice, since a launch
leaves the counters for the next."""
import numpy as np
import pytest

from flurrypp_amd import cases
from flurrypp_amd._native import PATH_FUSED, PATH_MIXED
from flurrypp_amd.batch import BatchedSolver, Member
from flurrypp_amd.solver import Solver
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu


# elements in flight in 128 blocks (quads) or 256 (hexes): quads 16384 (P0), 8192 (P1 to P5); hexes
# 32768 (P0, P1), 16384 (P2)
@pytest.mark.parametrize("kind,n,order,limit", [("vortex2d", 129, 0, 16384), ("vortex2d", 90, 1, 8192),
                                                ("vortex2d", 91, 1, 8192), ("vortex2d", 91, 3, 8192),
                                                ("vortex2d", 91, 5, 8192), ("vortex3d", 33, 0, 32768),
                                                ("vortex3d", 32, 1, 32768), ("vortex3d", 33, 1, 32768),
                                                ("vortex3d", 26, 2, 16384)])
def test_dt(kind, n, order, limit):
    setup, U = getattr(cases, kind)(n=n, order=order)
    print(f"{kind} {n} P{order}: {setup.nEles} elements, limit {limit}", flush=True)
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


def test_merged():
    """Three copies of a mesh in one context step as the mesh alone."""
    setup, U = cases.vortex2d(n=61, order=2)
    states = []
    for m in (1, 3):
        b = BatchedSolver([Member(setup, U) for _ in range(m)], path=PATH_FUSED)
        b.step(3)
        states += b.states()
        b.close()
    for st in states[1:]:
        # both forms of the stage kernel, whose sums are contracted differently at most
        np.testing.assert_allclose(st, states[0], rtol=1e-13, atol=1e-13)
