"""Inviscid steps of an odd number of stages, which end with U at the flux
points in the other of its two copies.  Wave speeds of single-stage steps with a
CFL time step: formed (and on the first step refreshed) before the time step, and
left there for the caller.  Against the oracle, after the first step and later
ones."""
import numpy as np
import pytest

from flurrypp_amd import cases
from flurrypp_amd._native import PATH_FUSED, PATH_MIXED, PATH_STAGED
from flurrypp_amd.mesh import pmg_operators
from flurrypp_amd.solver import MultiGrid, Solver
from oracle.oracle import Oracle, pmg_cycle

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


def _stages(setup, n):
    """Euler's step, or a three-stage one of the classical form."""
    p, fp = setup.params, setup.fp
    p.nRKSteps = fp.n_rk_steps = n
    p.RKa, p.RKb = ([0.0], [1.0]) if n == 1 else ([0.0, 0.5, 1.0], [1 / 6, 2 / 3, 1 / 6])
    for i in range(n):
        fp.rk_a[i], fp.rk_b[i] = p.RKa[i], p.RKb[i]


@pytest.mark.parametrize("path", [PATH_FUSED, PATH_MIXED])
def test_launches_of_a_step(path):
    """A single-stage step is the wave speeds with the time step, and the stage."""
    setup, U = CASES["bump2d"](2)
    s = Solver(setup.params, setup=setup)
    s.initializeSolution(U)
    s.update(1, path=path)
    s.enable_timing(True)
    s.update(4, path=path)
    n = {k.split("_", 1)[1]: v[1] for k, v in s.kernel_times().items()}
    s.close()
    assert n == {"extrapolate": 1, "wave_dt": 4, "stage": 4}


@pytest.mark.parametrize("path", [PATH_FUSED, PATH_MIXED])
@pytest.mark.parametrize("stages", [1, 3])
def test_replays(stages, path):
    """Steps in calls of other lengths (graphs of both copies) and one by one without graphs."""
    from flurrypp_amd import _native as nat
    runs = []
    for graphs in (1, 0):
        setup, U = cases.bump2d(nx=9, ny=5, order=2, cfl=0.2)
        _stages(setup, stages)
        s = Solver(setup.params, setup=setup)
        nat.hip_check(nat.hip_lib().fhip_set_option(s._ctx, 1, graphs))
        s.initializeSolution(U)
        out = []
        for n in ((1, 4, 3, 2, 5, 5) if graphs else (1,) * 20):
            s.update(n, path=path)
            out.append(s.get_U())
        runs.append([out[0], out[1], out[5]] if graphs else [out[0], out[4], out[19]])
        s.close()
    for a, b in zip(*runs):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("path,tol", [(PATH_FUSED, 1e-12), (PATH_MIXED, 1e-6)])
@pytest.mark.parametrize("stages,smooth", [(1, 1), (1, 2), (3, 1), (3, 2)])
@pytest.mark.parametrize("dt_type", [1, 2])
def test_multigrid(stages, smooth, dt_type, path, tol):
    """Cycles whose smoothing leaves either copy current, replayed from the third on."""
    setup, U = cases.bump2d(nx=10, ny=4, order=3, dt_type=dt_type, cfl=0.2)
    _stages(setup, stages)
    fine = Solver(setup.params, setup=setup)
    fine.initializeSolution(U)
    mg = MultiGrid(fine, low_order=0, smooth_steps=smooth)
    for s in mg.coarse:
        assert s._fp.n_rk_steps == stages
    ors = []
    for s in mg.levels:
        o = Oracle.from_setup(s.host)
        o.initializeSolution(s.host.initial_condition() if s is not fine else U, s.params.dtType)
        ors.append(o)
    R = [pmg_operators(2, s.order)[1] for s in mg.levels[1:]]
    Pr = [pmg_operators(2, s.order)[0] for s in mg.levels[:-1]]
    for _ in range(4):
        fine.update(1, path=path)
        mg.cycle(path)
        ors[-1].update(1)
        pmg_cycle(ors, R, Pr, smooth)
    # the bars of the multigrid tests
    for s, o in zip(mg.levels, ors):
        assert np.linalg.norm(s.get_U() - o.get_U()) <= tol * np.linalg.norm(o.get_U()), s.order
    mg.close()
    fine.close()


def _euler_step(setup):
    setup.params.timeType = setup.fp.time_type = 0
    _stages(setup, 1)


@pytest.mark.parametrize("path", [PATH_FUSED, PATH_MIXED])
@pytest.mark.parametrize("make", [
    lambda: cases.bump2d(nx=67, ny=61, order=3, dt_type=2, cfl=0.3),    # 4087 of 8 lanes: the last in 256 threads
    lambda: cases.bump2d(nx=69, ny=61, order=3, dt_type=1, cfl=0.3),    # 4209: blocks of 1024
    lambda: cases.vortex2d(n=91, order=3, cfl=0.3),                     # 132 k points: in two launches
    lambda: cases.vortex3d(n=4, order=3), lambda: cases.vortex3d(n=16, order=1),  # 4096 of 24 points, 2048 a turn
    lambda: cases.vortex3d(n=11, order=4)],
    ids=["quads_256", "quads_1024", "quads_apart", "hexes_256", "hexes_1024", "hexes_apart"])
def test_wave_speeds_and_time_steps(make, path):
    """The pass that forms both, at the edges of its block sizes and past its limit."""
    setup, U = make()
    _euler_step(setup)
    s, o = Solver(setup.params, setup=setup), Oracle.from_setup(setup)
    s.initializeSolution(U)
    o.initializeSolution(U, setup.params.dtType)
    for n in (1, 2):
        s.update(n, path=path)
        o.update(n)
        np.testing.assert_allclose(s.get("waveSp"), o.get("waveSp"), rtol=RTOL[path])
        # sums of the wave speeds: their bar
        np.testing.assert_allclose(s.get("ele_dt"), o.get("ele_dt"), rtol=RTOL[path])
        assert s.dt == s.get("ele_dt").min()
    s.close()
