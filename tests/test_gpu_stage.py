"""The stage kernel of inviscid runs (common flux, divergence, RK update and U
at the flux points in one launch) where it can go wrong: odd and even numbers
of stages (it reads one copy of U at the flux points and writes the other), a
time step taken from the residual it applies, the element time steps it forms
itself, blocks that hold parts of several elements, boundary faces with and
without Roe, residual-only launches between steps.  Against the oracle."""
import numpy as np
import pytest

from flurrypp_amd import cases
from flurrypp_amd._native import PATH_FUSED
from flurrypp_amd.solver import Solver
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu

TOL = 1e-12  # state after 10 steps, the bar of the parity tests


def _pair(setup, U):
    s, o = Solver(setup.params, setup=setup), Oracle.from_setup(setup)
    s.initializeSolution(U)
    o.initializeSolution(U, setup.params.dtType)
    return s, o


def _check(s, o):
    err = float(np.linalg.norm(s.get_U() - o.get_U()) / np.linalg.norm(o.get_U()))
    print(f"rel_l2={err:.3e}", flush=True)
    assert err < TOL
    np.testing.assert_allclose(s.get("waveSp"), o.get("waveSp"), rtol=1e-11)


def _three_stages(setup):
    """RK coefficients of a three-stage scheme (classical form)."""
    p, fp = setup.params, setup.fp
    p.nRKSteps = fp.n_rk_steps = 3
    p.RKa, p.RKb = [0.0, 0.5, 1.0], [1 / 6, 2 / 3, 1 / 6]
    for i, v in enumerate(p.RKa):
        fp.rk_a[i] = v
    for i, v in enumerate(p.RKb):
        fp.rk_b[i] = v


@pytest.mark.parametrize("dt_type", [0, 1, 2])
@pytest.mark.parametrize("time_type,stages", [(0, 1), (2, 2), (4, 3), (4, 4), (5, 4), (6, 4)])
def test_stages_and_time_steps(dt_type, time_type, stages):
    setup, U = cases.bump2d(nx=9, ny=5, order=2, dt_type=dt_type, time_type=time_type, cfl=0.3)
    if stages == 3:
        _three_stages(setup)
    s, o = _pair(setup, U)
    for n in (1, 4, 5):
        s.update(n, path=PATH_FUSED)
        o.update(n)
    _check(s, o)
    if dt_type == 2:
        np.testing.assert_allclose(s.get("ele_dt"), o.get("ele_dt"), rtol=1e-12)
    s.close()


@pytest.mark.parametrize("order", range(6))
@pytest.mark.parametrize("nt", [64, 192, 320])
def test_blocks_of_every_order(order, nt):
    setup, U = cases.bump2d(nx=7, ny=3, order=order, cfl=0.3)
    s, o = _pair(setup, U)
    s.set_block_sizes([256, 64, nt, 64, 256], PATH_FUSED) if order else None
    s.update(10, path=PATH_FUSED)
    o.update(10)
    _check(s, o)
    s.close()


@pytest.mark.parametrize("n,order", [(33, 0), (67, 3), (112, 1)])
def test_both_forms_agree(n, order):
    """Solution and flux points in threads of their own (small meshes) and in the
    same threads: the same state, on either side of the size where one takes
    over."""
    states = []
    for m in (1, 3):  # copies of one mesh merged into a context: beyond the limit with three
        from flurrypp_amd.batch import BatchedSolver, Member
        setup, U = cases.bump2d(nx=n, ny=n // 2, order=order, cfl=0.3)
        b = BatchedSolver([Member(setup, U) for _ in range(m)], path=PATH_FUSED)
        b.step(3)
        states += b.states()
        b.close()
    for st in states[1:]:
        np.testing.assert_allclose(st, states[0], rtol=1e-13, atol=1e-14)


@pytest.mark.parametrize("order", [0, 1, 3])
def test_hexes(order):
    setup, U = cases.tgv3d(n=3, order=order, viscous=0, jitter=0.1)
    s, o = _pair(setup, U)
    s.update(10, path=PATH_FUSED)
    o.update(10)
    _check(s, o)
    s.close()
