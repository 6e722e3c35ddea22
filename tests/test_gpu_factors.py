"""Operators of the fused kernels by their 1-D factors and from per-point tables
(the fallback for operators with the same non-zeros but other values): rows
scaled point by point have no common factors, so the tables are read.  Against
the oracle with the same operators."""
import numpy as np
import pytest

from flurrypp_amd import cases
from flurrypp_amd._native import PATH_FUSED, PATH_MIXED
from flurrypp_amd.solver import Solver
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu


def _scaled(setup, names):
    """Every row of the operators scaled by its own factor near one."""
    rng = np.random.default_rng(5)
    for name in names:
        a = getattr(setup.opers, name)
        f = 1.0 + 1e-3 * rng.uniform(-1.0, 1.0, a.shape[:-1])
        setattr(setup.opers, name, np.ascontiguousarray(a * f[..., None]))


CASES = {
    "vortex2d_p1": (lambda: cases.vortex2d(n=5, order=1), ("spts_to_fpts", "correction")),
    "bump2d_p3": (lambda: cases.bump2d(nx=7, ny=3, order=3, cfl=0.3), ("correction",)),
    "bump2d_p4": (lambda: cases.bump2d(nx=7, ny=3, order=4, cfl=0.3), ("spts_to_fpts", "extrap_fn")),
    "tgv3d_p2_ns": (lambda: cases.tgv3d(n=3, order=2, viscous=1, jitter=0.1), ("correct_u", "correction")),
    "tgv3d_p3_ns": (lambda: cases.tgv3d(n=3, order=3, viscous=1, jitter=0.1), ("spts_to_fpts", "correct_u")),
    "tgv3d_p3_euler": (lambda: cases.tgv3d(n=3, order=3, viscous=0, jitter=0.1), ("correction",)),
}


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("scaled", [False, True])
def test_factors_and_tables(name, scaled):
    make, ops = CASES[name]
    setup, U = make()
    if scaled:
        _scaled(setup, ops)
    s, o = Solver(setup.params, setup=setup), Oracle.from_setup(setup)
    assert s._fused_ok()
    o.initializeSolution(U, setup.params.dtType)
    o.update(6)
    # the parity bars: 1e-12 for the FP64 state after 10 steps, 1e-6 for the mixed one
    for path, tol in ((PATH_FUSED, 1e-12), (PATH_MIXED, 1e-6)):
        t = Solver(setup.params, setup=setup)
        t.initializeSolution(U)
        t.update(6, path=path)
        err = float(np.linalg.norm(t.get_U() - o.get_U()) / np.linalg.norm(o.get_U()))
        print(f"{name} scaled={scaled} path={path} rel_l2={err:.3e}", flush=True)
        assert err < tol
        t.close()
    s.close()
