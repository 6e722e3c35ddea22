"""The viscous volume kernel at low orders, where an element takes a thread per
flux point and its solution points the first of them: quads and hexes, walls and
none, blocks that hold part of a mesh's elements or more than all, both
precisions.  Against the oracle."""
import numpy as np
import pytest

from flurrypp_amd import cases
from flurrypp_amd._native import PATH_FUSED, PATH_MIXED
from flurrypp_amd.input import InputParams
from flurrypp_amd.mesh import Mesh
from flurrypp_amd.solver import HostSetup, Solver
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu

# the parity bars: 1e-12 for the FP64 state after 10 steps, 1e-6 for the mixed one
PATHS = ((PATH_FUSED, 1e-12), (PATH_MIXED, 1e-6))


def _walls(nx, ny, order, nz=0):
    """A box with no-slip walls, adiabatic or at a temperature, and characteristic ends."""
    d = dict(equation=1, nDims=3 if nz else 2, order=order, meshType=1, nx=nx, ny=ny, nz=max(nz, 1), xmin=0, xmax=1, ymin=0,
             ymax=1, zmin=0, zmax=1, timeType=4, dtType=1, CFL=0.4, maxTime=1e9, iterMax=10, icType=0, viscous=1,
             Re=100, MachBound=0.3, MachWall=0.1, fixVis=0, LDG_penFact=0.5, LDG_tau=1.0, TWall=320.0)
    p = InputParams.from_dict(d)
    bcs = {"left": "char", "right": "char", "bottom": "adiabatic_noslip", "top": "isothermal_noslip_moving"}
    if nz:
        bcs.update(front="isothermal_noslip", back="slip_wall")
        m = Mesh.cartesian(3, (nx, ny, nz), (0, 0, 0), (1, 1, 1), bcs=bcs)
    else:
        m = Mesh.cartesian(2, (nx, ny), (0, 0), (1, 1), bcs=bcs)
    s = HostSetup(p, m)
    U = s.initial_condition()
    return s, U * (1 + 0.01 * np.sin(np.arange(U.size)).reshape(U.shape))


def _check(setup, U, nt, path, tol, steps=10):
    o = Oracle.from_setup(setup)
    o.initializeSolution(U, setup.params.dtType)
    s = Solver(setup.params, setup=setup)
    s.initializeSolution(U)
    if nt:
        s.set_block_sizes([256, 64, nt, 64, 64], path)
    s.update(steps, path=path)
    o.update(steps)
    err = float(np.linalg.norm(s.get_U() - o.get_U()) / np.linalg.norm(o.get_U()))
    print(f"P{setup.order} {setup.nEles} elements nt={nt} path={path} rel_l2={err:.3e}", flush=True)
    assert err < tol
    if path == PATH_FUSED:
        np.testing.assert_allclose(s.get("waveSp"), o.get("waveSp"), rtol=1e-11)
    s.close()


@pytest.mark.parametrize("path,tol", PATHS)
@pytest.mark.parametrize("nt", [64, 100, 192, 0])
@pytest.mark.parametrize("nx,ny,order", [(1, 1, 0), (13, 7, 0), (1, 2, 1), (9, 5, 1), (7, 3, 2), (16, 8, 2)])
def test_quads(nx, ny, order, nt, path, tol):
    setup, U = _walls(nx, ny, order)
    _check(setup, U, nt, path, tol)


@pytest.mark.parametrize("path,tol", PATHS)
@pytest.mark.parametrize("nt", [64, 100, 0])
@pytest.mark.parametrize("n,order", [(1, 0), (4, 0), (1, 1), (3, 1)])
def test_hexes(n, order, nt, path, tol):
    setup, U = _walls(n, n + 1, order, n + 2)
    _check(setup, U, nt, path, tol)


@pytest.mark.parametrize("path,tol", PATHS)
@pytest.mark.parametrize("order", [0, 1, 2])
def test_periodic(order, path, tol):
    """No boundary points: the other instances."""
    setup, U = cases.tgv3d(n=3, order=order, viscous=1, jitter=0.1)
    _check(setup, U, 0, path, tol)


@pytest.mark.parametrize("path,tol", PATHS)
def test_largest_block(path, tol):
    """P1 quads at 512 threads: the size whose LDS was at the limit."""
    setup, U = _walls(19, 7, 1)
    _check(setup, U, 512, path, tol)
