"""Both forms of the inviscid stage kernel (solution and flux points in threads
of their own, and in the same threads), on either side of the size where one
takes over: E * (S + F) of 64 lanes * 4096 waves for quads (P0 has but one form).  Copies of one mesh
merged into a context reach it; the element counts say which side each is on."""
import numpy as np
import pytest

from flurrypp_amd import cases
from flurrypp_amd._native import PATH_FUSED, PATH_MIXED
from flurrypp_amd.batch import BatchedSolver, Member
from flurrypp_amd.mesh import pmg_operators
from flurrypp_amd.solver import MultiGrid, Solver
from oracle.oracle import Oracle, pmg_cycle

pytestmark = pytest.mark.gpu

LIMIT = 4096 * 64  # lanes of the quads' apart form


def _apart(setup, copies=1):
    return copies * setup.nEles * (setup.nSpts + setup.nFpts) <= LIMIT


@pytest.mark.parametrize("path,rtol", [(PATH_FUSED, 1e-13), (PATH_MIXED, 1e-6)])
@pytest.mark.parametrize("dt_type", [1, 2])
@pytest.mark.parametrize("nx,ny,order,copies", [(160, 101, 1, 2), (101, 83, 2, 2), (67, 33, 3, 5),
                                                (60, 61, 4, 2), (45, 53, 5, 2)])
def test_both_forms_agree(nx, ny, order, copies, dt_type, path, rtol):
    setup, U = cases.bump2d(nx=nx, ny=ny, order=order, cfl=0.3, dt_type=dt_type)
    assert _apart(setup) and not _apart(setup, copies)
    print(f"P{order} {setup.nEles} elements, {copies} copies", flush=True)
    states = []
    for m in (1, copies):
        b = BatchedSolver([Member(setup, U) for _ in range(m)], path=path)
        b.step(3)
        states += b.states()
        b.close()
    for st in states[1:]:
        # sums of the same terms in the same order, contracted differently at most
        np.testing.assert_allclose(st, states[0], rtol=rtol, atol=rtol)


@pytest.mark.parametrize("time_type,dt_type", [(6, 2), (4, 2), (4, 0)])
def test_multigrid_beyond_the_limit(time_type, dt_type):
    """A fine level and a coarse one past the limit: residuals, the source taken
    in the first smoothing stage, local time steps."""
    setup, U = cases.bump2d(nx=161, ny=80, order=3, time_type=time_type, dt_type=dt_type, dt=1e-4, cfl=0.5)
    fine = Solver(setup.params, setup=setup)
    fine.initializeSolution(U)
    mg = MultiGrid(fine, low_order=1, smooth_steps=2)
    assert not _apart(fine.host) and not _apart(mg.coarse[-1].host) and _apart(mg.coarse[0].host)
    ors = []
    for s in mg.levels:
        o = Oracle.from_setup(s.host)
        o.initializeSolution(s.host.initial_condition() if s is not fine else U, s.params.dtType)
        ors.append(o)
    R = [pmg_operators(2, s.order)[1] for s in mg.levels[1:]]
    Pr = [pmg_operators(2, s.order)[0] for s in mg.levels[:-1]]
    for _ in range(2):
        fine.update(1, path=PATH_FUSED)
        mg.cycle(PATH_FUSED)
        ors[-1].update(1)
        pmg_cycle(ors, R, Pr, 2)
    for s, o in zip(mg.levels, ors):
        err = float(np.linalg.norm(s.get_U() - o.get_U()) / np.linalg.norm(o.get_U()))
        print(f"P{s.order} rel_l2={err:.3e}", flush=True)
        assert err < 1e-12  # the bar of the multigrid tests
    mg.close()
    fine.close()


@pytest.mark.parametrize("nx,ny,nt", [(29, 13, 64), (29, 13, 192), (29, 13, 256), (241, 223, 0)])
def test_p0(nx, ny, nt):
    """P0 quads at block sizes other than the default, and more of them than other
    orders keep apart, against the oracle."""
    setup, U = cases.bump2d(nx=nx, ny=ny, order=0, cfl=0.3)
    s, o = Solver(setup.params, setup=setup), Oracle.from_setup(setup)
    s.initializeSolution(U)
    o.initializeSolution(U, setup.params.dtType)
    if nt:
        s.set_block_sizes([256, 64, nt, 64, 256], PATH_FUSED)
    s.update(10, path=PATH_FUSED)
    o.update(10)
    assert np.linalg.norm(s.get_U() - o.get_U()) < 1e-12 * np.linalg.norm(o.get_U())
    s.close()
