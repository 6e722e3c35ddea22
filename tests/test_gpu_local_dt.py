"""The solver's dt with local time steps (dt_type 2): the smallest of the
elements' time steps, as solver::calcDt leaves it (src/solver.cpp:447-468),
after every call that took a step: updates of one and several stages, one
block and several of elements, both precisions, multigrid levels, the main
loop's time.  Against the oracle."""
import numpy as np
import pytest

from flurrypp_amd import cases
from flurrypp_amd._native import PATH_FUSED, PATH_MIXED, PATH_STAGED
from flurrypp_amd.input import InputParams
from flurrypp_amd.mesh import pmg_operators
from flurrypp_amd.solver import HostSetup, MultiGrid, Solver, run
from oracle.oracle import Oracle, pmg_cycle

pytestmark = pytest.mark.gpu

# the parity tests' bars for dt on the FP64 paths and on the mixed one
RTOL = {PATH_FUSED: 1e-12, PATH_STAGED: 1e-12, PATH_MIXED: 1e-6}


def _pair(setup, U):
    s, o = Solver(setup.params, setup=setup), Oracle.from_setup(setup)
    s.initializeSolution(U)
    o.initializeSolution(U, setup.params.dtType)
    return s, o


@pytest.mark.parametrize("path", [PATH_FUSED, PATH_MIXED, PATH_STAGED])
@pytest.mark.parametrize("nx,ny,order,time_type", [(3, 1, 1, 4), (9, 5, 2, 0), (9, 5, 2, 4), (9, 5, 2, 6),
                                                   (32, 8, 0, 4), (41, 25, 1, 4), (101, 61, 2, 6)])
def test_update(nx, ny, order, time_type, path):
    setup, U = cases.bump2d(nx=nx, ny=ny, order=order, time_type=time_type, cfl=0.3)
    s, o = _pair(setup, U)
    for n in (1, 1, 3):
        s.update(n, path=path)
        o.update(n)
        print(f"dt {s.dt:.17e} oracle {o.dt:.17e}", flush=True)
        np.testing.assert_allclose(s.dt, o.dt, rtol=RTOL[path])
        assert s.dt == s.get("ele_dt").min()
    s.close()


@pytest.mark.parametrize("path", [PATH_FUSED, PATH_MIXED])
def test_replayed_steps(path):
    """Single steps, which replay one captured graph: dt follows the state."""
    setup, U = cases.bump2d(nx=41, ny=25, order=2, cfl=0.3)
    s, o = _pair(setup, U)
    seen = set()
    for _ in range(6):
        s.update(1, path=path)
        o.update(1)
        np.testing.assert_allclose(s.dt, o.dt, rtol=RTOL[path])
        seen.add(s.dt)
    assert len(seen) > 1
    s.close()


@pytest.mark.parametrize("path", [PATH_FUSED, PATH_MIXED, PATH_STAGED])
def test_multigrid_levels(path):
    """Every coarse level's dt is its last smoothing step's; a cycle leaves the
    fine level's as it was, also where a caller has set it."""
    setup, U = cases.bump2d(nx=41, ny=25, order=3, time_type=6, cfl=0.9)
    fine = Solver(setup.params, setup=setup)
    fine.initializeSolution(U)
    mg = MultiGrid(fine, low_order=0, smooth_steps=2)
    ors = []
    for s in mg.levels:
        o = Oracle.from_setup(s.host)
        o.initializeSolution(s.host.initial_condition() if s is not fine else U, s.params.dtType)
        ors.append(o)
    R = [pmg_operators(2, s.order)[1] for s in mg.levels[1:]]
    Pr = [pmg_operators(2, s.order)[0] for s in mg.levels[:-1]]
    for _ in range(4):
        fine.update(1, path=path)
        ors[-1].update(1)
        np.testing.assert_allclose(fine.dt, ors[-1].dt, rtol=RTOL[path])
        fine.set_dt(0.125)
        mg.cycle(path)
        pmg_cycle(ors, R, Pr, 2)
        assert fine.dt == 0.125
        for s, o in zip(mg.coarse, ors):
            np.testing.assert_allclose(s.dt, o.dt, rtol=RTOL[path])
    mg.close()
    fine.close()


def test_no_step_leaves_dt():
    """update(0) and a cycle without smoothing take no step."""
    setup, U = cases.bump2d(nx=9, ny=5, order=2, time_type=6, cfl=0.9)
    fine = Solver(setup.params, setup=setup)
    fine.initializeSolution(U)
    mg = MultiGrid(fine, low_order=0, smooth_steps=0)
    for s in mg.levels:
        s.set_dt(0.25)
    fine.update(0, path=PATH_FUSED)
    for _ in range(3):
        mg.cycle(PATH_FUSED)
    assert [s.dt for s in mg.levels] == [0.25] * 3
    mg.close()
    fine.close()


def test_run():
    """The main loop of an input file with dtType 2: the time advances by dt."""
    d = dict(equation=1, nDims=2, order=2, meshType=1, nx=6, ny=6, xmin=-5, xmax=5, ymin=-5, ymax=5, timeType=4,
             dtType=2, CFL=0.5, maxTime=1e9, iterMax=5, icType=2, monitorResFreq=2, plotFreq=1000, resType=2)
    p = InputParams.from_dict(d)
    s = run(p, log=lambda line: None, output_dir=None)
    assert s.iter == 5
    s.close()
    setup = HostSetup(InputParams.from_dict(d))
    o = Oracle.from_setup(setup)
    o.initializeSolution(setup.initial_condition(), 2)
    time = 0.0
    for _ in range(5):
        o.update(1)
        time += o.dt
    np.testing.assert_allclose(p.time, time, rtol=1e-12)
