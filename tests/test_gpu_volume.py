"""The volume kernel of viscous runs (common flux and LDG common U of the element's
own flux points, all of the residual but the other sides' LDG parts) where it can
go wrong: every order, blocks that hold parts of several elements, threads with
several flux points and with none, time steps from its wave speeds, single-stage
steps, both precisions.  Against the oracle."""
import numpy as np
import pytest

from flurrypp_amd import cases
from flurrypp_amd._native import PATH_FUSED, PATH_MIXED
from flurrypp_amd.solver import Solver
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu

# the parity bars: 1e-12 for the FP64 state after 10 steps, 1e-6 for the mixed one
PATHS = ((PATH_FUSED, 1e-12), (PATH_MIXED, 1e-6))


def _check(setup, U, blocks=None, steps=10):
    o = Oracle.from_setup(setup)
    o.initializeSolution(U, setup.params.dtType)
    o.update(steps)
    for path, tol in PATHS:
        s = Solver(setup.params, setup=setup)
        s.initializeSolution(U)
        if blocks:
            s.set_block_sizes(blocks, path)
        s.update(steps, path=path)
        err = float(np.linalg.norm(s.get_U() - o.get_U()) / np.linalg.norm(o.get_U()))
        print(f"P{setup.order} blocks={blocks} path={path} rel_l2={err:.3e}", flush=True)
        assert err < tol
        if path == PATH_FUSED:
            np.testing.assert_allclose(s.get("waveSp"), o.get("waveSp"), rtol=1e-11)
        s.close()


@pytest.mark.parametrize("order,nt", [(0, 64), (0, 128), (1, 64), (1, 192), (2, 64), (2, 320), (3, 64), (3, 256),
                                      (4, 128), (4, 320), (5, 256), (5, 384)])
def test_blocks_of_every_order(order, nt):
    setup, U = cases.tgv3d(n=3, order=order, viscous=1, jitter=0.1)
    _check(setup, U, [256, 64, nt, 64, max(nt, 64 if order else 64)])


@pytest.mark.parametrize("time_type", [0, 4])
@pytest.mark.parametrize("dt_type", [1, 2])
def test_time_steps(time_type, dt_type):
    setup, U = cases.tgv3d(n=3, order=2, viscous=1, jitter=0.1)
    setup.params.timeType, setup.params.dtType, setup.params.CFL = time_type, dt_type, 0.3
    setup.fp.time_type, setup.fp.dt_type, setup.fp.cfl = time_type, dt_type, 0.3
    if time_type == 0:
        p = setup.params
        p.nRKSteps = setup.fp.n_rk_steps = 1
        p.RKa, p.RKb = [0.0], [1.0]
        setup.fp.rk_a[0], setup.fp.rk_b[0] = 0.0, 1.0
    _check(setup, U, steps=5)
