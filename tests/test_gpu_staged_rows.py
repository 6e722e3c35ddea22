"""Operators of the staged path by their non-zeros (k_oprows) and dense
(k_opgemm): orders above the fused paths' range, whose rows take the widest
form, and operators without zeros, which stay dense.  Against the oracle,
which multiplies every operator out."""
import numpy as np
import pytest

from flurrypp_amd import cases
from flurrypp_amd._native import PATH_STAGED
from flurrypp_amd.solver import Solver
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu

# sums of at most 3 * 64 products of like terms: 192 roundings of 1.1e-16, against the largest of
# the arrays that the sums combine
TOL = 2.2e-14


def _dense(setup):
    """Every operator entry non-zero: the exact ones plus a small seeded remainder."""
    rng = np.random.default_rng(3)
    o = setup.opers
    for name in ("spts_to_fpts", "grad_spts", "extrap_fn", "correction", "correct_u"):
        a = getattr(o, name)
        setattr(o, name, np.ascontiguousarray(a + 1e-3 * rng.uniform(0.5, 1.0, a.shape)))


@pytest.mark.parametrize("order,dense", [(6, False), (10, False), (3, True), (4, True)])
def test_residual_2d(order, dense):
    setup, U = cases.vortex2d(n=3, order=order, dt_type=0)
    if dense:
        _dense(setup)
    _compare(setup, U)


@pytest.mark.parametrize("order,dense", [(1, False), (6, False), (3, True)])
def test_residual_3d_viscous(order, dense):
    setup, U = cases.tgv3d(n=3, order=order, viscous=1, dt=1e-4, jitter=0.1)
    if dense:
        _dense(setup)
    _compare(setup, U)


def _compare(setup, U):
    s, o = Solver(setup.params, setup=setup), Oracle.from_setup(setup)
    assert s.params.order > 5 or s._fused_ok() == (setup.opers.spts_to_fpts == 0).any()
    s.initializeSolution(U)
    o.initializeSolution(U, 0)
    s.calcResidual(0)
    o.calcResidual(0)
    scale = {"disFn_fpts": "Fn_fpts", "divF_spts": "F_spts", "dU_spts": "U_spts", "dU_fpts": "U_fpts"}
    for a in ["U_fpts", "F_spts", "disFn_fpts", "divF_spts"] + (["dU_spts", "dU_fpts"] if s.params.viscous else []):
        ref = o.get(a)
        den = max(np.linalg.norm(ref), np.linalg.norm(o.get(scale[a])) if a in scale else 0.0)
        err = float(np.linalg.norm(s.get(a) - ref) / den)
        print(f"{a} rel_l2={err:.3e}", flush=True)
        assert err < TOL, a
    s.update(2, path=PATH_STAGED)
    o.update(2)
    assert np.linalg.norm(s.get_U() - o.get_U()) <= 1e-13 * np.linalg.norm(o.get_U())
    s.close()
