"""Tuned block sizes are shared by contexts that run the same kernels: of meshes
in one power of two of the element count, those on the other side of the size
where the inviscid stage kernel changes its form are tuned by themselves, and so
are operators that are read from tables."""
import numpy as np
import pytest

from flurrypp_amd import cases
from flurrypp_amd._native import PATH_FUSED, PATH_MIXED, PATH_MIXED_BF16, PATH_MIXED_BF16X3
from flurrypp_amd.solver import Solver

pytestmark = pytest.mark.gpu


def _tunes(nx, ny, scaled=False):
    """Whether autotune timed kernels (it starts with an extrapolation), rather than
    take sizes found before."""
    setup, U = cases.bump2d(nx=nx, ny=ny, order=5, cfl=0.3)
    if scaled:  # rows of their own: no common 1-D factors
        a = setup.opers.correction
        setup.opers.correction = np.ascontiguousarray(a * (1.0 + 1e-3 * np.arange(a.shape[0]))[:, None])
    s = Solver(setup.params, setup=setup)
    s.initializeSolution(U)
    s.enable_timing(True)
    s.autotune(PATH_MIXED)
    ran = "mixed_extrapolate" in s.kernel_times()
    s.close()
    return ran


def test_key():
    # P5 quads: apart up to 4096 * 64 / (36 + 24) = 4369 elements; all within 4096..8191
    _tunes(60, 70)                       # 4200, whatever ran before in this process
    assert not _tunes(61, 70)            # 4270: the same kernels
    assert _tunes(71, 70)                # 4970: the other form
    assert not _tunes(70, 70)
    assert _tunes(60, 70, scaled=True)   # tables
    assert not _tunes(61, 70, scaled=True)


def test_key_of_mixed_forms():
    """The BF16 forms of the mixed path are kernels of their own, and tuned by themselves."""
    def tunes(n, path):
        setup, U = cases.vortex3d(n=n, order=3)
        s = Solver(setup.params, setup=setup)
        s.initializeSolution(U)
        s.enable_timing(True)
        s.autotune(path)
        ran = "mixed_extrapolate" in s.kernel_times()
        s.close()
        return ran

    for path in (PATH_MIXED, PATH_MIXED_BF16, PATH_MIXED_BF16X3):
        tunes(4, path)          # 64 elements, whatever ran before in this process
    for path in (PATH_MIXED, PATH_MIXED_BF16, PATH_MIXED_BF16X3):
        assert not tunes(5, path)  # 125
    assert tunes(9, PATH_MIXED)             # 729
    assert tunes(9, PATH_MIXED_BF16)
    assert tunes(9, PATH_MIXED_BF16X3)
    assert not tunes(9, PATH_MIXED)


def test_sizes_by_path():
    """Sizes tuned or set for one fused path leave the other paths' sizes alone."""
    setup, U = cases.vortex3d(n=4, order=3)
    s = Solver(setup.params, setup=setup)
    s.initializeSolution(U)
    paths = (PATH_FUSED, PATH_MIXED, PATH_MIXED_BF16, PATH_MIXED_BF16X3)
    sizes = [[64 * (i + 1), 64, 64 * (i + 2), 64, 256] for i in range(4)]
    for path, nt in zip(paths, sizes):
        s.set_block_sizes(nt, path)
    for path, nt in zip(paths, sizes):
        assert s.block_sizes(path) == nt
    s.close()
