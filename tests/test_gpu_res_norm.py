"""The residual norm's reduction (blocks of 256 elements by groups of solution
points) at its edges: one element row short of, at and past a block, as many
points as groups and fewer, all three norms.  Against the oracle."""
import numpy as np
import pytest

from flurrypp_amd import cases
from flurrypp_amd.solver import Solver
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("make", [
    lambda: cases.vortex2d(n=3, order=0), lambda: cases.bump2d(nx=51, ny=5, order=1),
    lambda: cases.vortex2d(n=16, order=2), lambda: cases.bump2d(nx=257, ny=1, order=5),
    lambda: cases.tgv3d(n=7, order=3, jitter=0.1)])
def test_every_norm(make):
    setup, U = make()
    s, o = Solver(setup.params, setup=setup), Oracle.from_setup(setup)
    s.initializeSolution(U)
    o.initializeSolution(U, setup.params.dtType)
    s.update(2)
    o.update(2)
    for t in (1, 2, 3):
        # the bar of the parity tests' norm
        np.testing.assert_allclose(s.residual_norm(t), o.residual_norm(t), rtol=1e-10, atol=1e-13)
    s.close()
