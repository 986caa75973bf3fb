"""GPU parity of the single-iteration smoother (k_rb_fused, and k_rb_fused_down on every second iteration) against the
oracle on the levels it serves when no tile is set, between those smoothed by blocks and those by sweeps: FP64 bit for
bit, FP32 within the bound of the FP32 smoothers.  (test_vcycle_fp64_bitwise and test_mixed_precision_vs_fp64_oracle run
the tiles that are set; test_gpu_fp32_kernels_agree compares the FP32 ones with this route's values.)"""
import ctypes as C

import numpy as np
import pytest

from oracle import oracle as O
from peps_mg_amd import _lib, geometry, matrix
from peps_mg_amd.multigrid import Multigrid
from peps_mg_amd.rbgs_poisson_matrix import rbgs_iterator_fp32, rbgs_iterator_poisson_matrix

pytestmark = pytest.mark.gpu


def sdm_from(g):
    return geometry.Subdomain(g.nx, g.ny, g.nz, 0, 0, 0, g.sox, g.soy, g.soz, g.dxm, g.dym, g.dzm, g.dxg, g.dyg,
                              g.dzg, g.xg, g.yg, g.zg)


# partial tiles along x and y, odd plane counts (the top chunk ends on an even plane and the downward march starts one
# plane above the domain), odd rows; stretched where the axis is even
FP64 = [((70, 520, 37), (1.01, 1.003, 1.0), "64, 32"), ((130, 150, 71), (1.01, 1.01, 1.0), "64, 8"),
        ((171, 157, 51), (1.0, 1.0, 1.0), "64, 8"), ((128, 128, 128), (1.0, 1.0, 1.01), "64, 32"),
        # more large blocks than CUs: 300, 405 and 576
        ((80, 80, 80), (1.01, 1.0, 1.0), "64, 8"), ((131, 67, 69), (1.0, 1.0, 1.0), "64, 8"),
        ((96, 96, 128), (1.0, 1.01, 1.0), "64, 8")]


@pytest.mark.parametrize("dims,stretch,tile", FP64)
@pytest.mark.parametrize("omega,nu", [(1.0, 1), (1.6, 2), (1.0, 5)])
def test_fp64_bitwise(dims, stretch, tile, omega, nu):
    g = O.Grid(*dims, a=stretch)
    A = g.matrix()
    x, b = O.uniform_field(*dims, 81), O.uniform_field(*dims, 82)
    xg = x.copy()
    rbgs_iterator_poisson_matrix(xg, matrix.MatrixHeptadiagonal(0, A), b, sdm_from(g), nu, omega)
    O.rbgs_iterator(x, A, b, nu, omega)
    assert np.array_equal(xg, x)


FP32 = [((74, 1200, 37), (1.01, 1.002, 1.0), "128, 32"), ((128, 128, 200), (1.0, 1.0, 1.01), "128, 32"),
        ((200, 300, 53), (1.0, 1.005, 1.0), "128, 32"), ((171, 157, 117), (1.0, 1.0, 1.0), "64, 8"),
        ((162, 150, 130), (1.01, 1.0, 1.01), "64, 8")]


@pytest.mark.parametrize("dims,stretch,tile", FP32)
@pytest.mark.parametrize("omega,nu", [(1.0, 1), (1.35, 2), (1.6, 3)])
def test_fp32_against_oracle(dims, stretch, tile, omega, nu):
    """Bound: 1e-6 (1 + nu), relative to max|x| (a numpy FP32 emulation of the reference loop lands within 1.5e-6 of the
    FP64 iteration for up to 6 iterations)."""
    g = O.Grid(*dims, a=stretch)
    x = O.uniform_field(*dims, 83).astype(np.float32).astype(np.float64)
    b = O.uniform_field(*dims, 84).astype(np.float32).astype(np.float64)
    x32 = x.copy()
    rbgs_iterator_fp32(x32, b, sdm_from(g), nu, omega)
    O.rbgs_iterator(x, g.matrix(), b, nu, omega)
    assert np.array_equal(x32, x32.astype(np.float32).astype(np.float64))
    err = np.abs(x32 - x).max() / np.abs(x).max()
    assert err < 1e-6 * (1 + nu), err


@pytest.mark.parametrize("precision,dims,tile", [(0, d, t) for d, _, t in FP64] + [(1, d, t) for d, _, t in FP32])
def test_route(precision, dims, tile):
    """The grids above run the single-iteration kernel in the tile named (axes rounded down to two halvings)."""
    dims = tuple(n // 4 * 4 for n in dims)
    sdm = geometry.geometry_subdomain_create(geometry.geometry_domain_create(*dims, 0.0, 0.0, 0.0, 1.0, 1.0, 1.0))
    mg = Multigrid(sdm, 2, 1, precision=precision)
    avg, nb, kn = C.c_double(0), C.c_double(0), C.c_char_p()
    _lib.check(_lib.lib().pepsmg_bench_smoother(mg.h, precision, 1, 1.0, C.byref(avg), C.byref(nb), C.byref(kn)))
    mg.destroy()
    assert kn.value.decode() == f"k_rb_fused<{'float' if precision else 'double'}, {tile}, 0, 1>"
