"""GPU parity of the two-iterations-a-pass smoother (k_sweep) against the oracle, on grids large enough that
it is the one the solver runs: FP64 bit for bit, FP32 within the bound of the single-iteration FP32 smoother.

The grids put the edges of tiles (128 x 32 cells with a ring of 4), of waves (4 rows) and of z-chunks inside
and at the faces of the level: whole tiles, partial tiles on every axis, odd cell counts (a pair with one cell
inside), a z axis whose coefficients differ from plane to plane (no kept divisors) and one row of tiles."""
import ctypes as C

import numpy as np
import pytest

from oracle import oracle as O
from peps_mg_amd import _lib, geometry, matrix
from peps_mg_amd.multigrid import Multigrid
from peps_mg_amd.rbgs_poisson_matrix import rbgs_iterator_fp32, rbgs_iterator_poisson_matrix

pytestmark = pytest.mark.gpu

GRIDS = [((128, 128, 256), (1.0, 1.0, 1.0)), ((170, 158, 156), (1.01, 1.0, 1.0)), ((171, 157, 153), (1.0, 1.0, 1.0)),
         ((250, 130, 128), (1.0, 1.004, 1.01)), ((512, 32, 256), (1.0, 1.0, 1.0))]
IDS = ["whole-x", "partial", "odd", "stretched-z", "one-row-of-tiles"]


def sdm_from(g):
    return geometry.Subdomain(g.nx, g.ny, g.nz, 0, 0, 0, g.sox, g.soy, g.soz, g.dxm, g.dym, g.dzm, g.dxg, g.dyg,
                              g.dzg, g.xg, g.yg, g.zg)


def field(dims, seed):
    return O.uniform_field(*dims, seed)


@pytest.mark.parametrize("dims,stretch", GRIDS, ids=IDS)
@pytest.mark.parametrize("omega,nu", [(1.0, 2), (1.6, 3), (1.0, 4)])
def test_iterator_fp64_bitwise(dims, stretch, omega, nu):
    g = O.Grid(*dims, a=stretch)
    A = g.matrix()
    x, b = field(dims, 3), field(dims, 4)
    b[5, 5:90, 1:] = 0.0                      # zero and tiny differences leave the kept divisors for a division
    x[3:8, 3:92, :] = 0.0
    b[20, 2, 1:9] = 1e-290
    xg = x.copy()
    rbgs_iterator_poisson_matrix(xg, matrix.MatrixHeptadiagonal(0, A), b, sdm_from(g), nu, omega)
    O.rbgs_iterator(x, A, b, nu, omega)
    assert np.array_equal(xg, x)


@pytest.mark.parametrize("dims,stretch", GRIDS, ids=IDS)
@pytest.mark.parametrize("omega,nu", [(1.0, 2), (1.35, 4)])
def test_iterator_fp32_against_oracle(dims, stretch, omega, nu):
    """The FP32 inner smoother from FP32-representable inputs; the bound 1e-6 (1 + nu), relative to max|x|, is
    the one of the single-iteration kernels (a numpy FP32 emulation of the reference loop lands within 1.5e-6
    of the FP64 iteration over 6 iterations; this kernel rounds less often)."""
    g = O.Grid(*dims, a=stretch)
    A = g.matrix()
    x = field(dims, 5).astype(np.float32).astype(np.float64)
    b = field(dims, 6).astype(np.float32).astype(np.float64)
    x32 = x.copy()
    rbgs_iterator_fp32(x32, b, sdm_from(g), nu, omega)
    O.rbgs_iterator(x, A, b, nu, omega)
    assert np.array_equal(x32, x32.astype(np.float32).astype(np.float64))
    err = np.abs(x32 - x).max() / np.abs(x).max()
    assert err < 1e-6 * (1 + nu), err


@pytest.mark.parametrize("dims,stretch,nlevel", [((176, 160, 144), (1.0, 1.0, 1.0), 4),
                                                 ((176, 160, 144), (1.004, 1.003, 1.005), 4)], ids=["uniform", "stretched"])
@pytest.mark.parametrize("nu", [2, 3])
def test_vcycle_large_ragged(dims, stretch, nlevel, nu):
    """Whole solves whose fine level runs k_sweep (mixed precision: also from 0 and after the prolongation), with
    partial tiles on every axis: FP64 bit-identical to the oracle; mixed precision with the residual it reports."""
    g = O.Grid(*dims, l=(1.1, 1.0, 0.9), a=stretch)
    A = g.matrix()
    b = field(dims, 7)
    mo = O.Multigrid(g, nlevel, 60)
    xo, ro = O.padded(*dims), O.padded(*dims)
    nc, hist, cit, res0 = mo.solve_vcycle(xo, ro, A, b, nu, 1e-10, 1.0)
    for precision in (0, 1):
        mg = Multigrid(sdm_from(g), nlevel, 60, precision=precision)
        x, r = O.padded(*dims), O.padded(*dims)
        res = mg.solve_vcycle(x, r, None, b, nu, 1e-10, 1.0)
        assert res.converged
        if precision == 0:
            assert res.cycles == nc and np.array_equal(x, xo) and np.array_equal(r, ro)
        else:
            # the reported residual is the one an FP64 evaluation of b - A x gives, and below the tolerance
            rr = (b - O.mv_mul(A, x))[1:-1, 1:-1, 1:-1]
            rho = np.sqrt(np.sum(rr * rr) / res.res0)
            assert rho < 1e-10 and abs(rho - res.rho) <= 1e-3 * res.rho
        avg, nb, kn = C.c_double(0), C.c_double(0), C.c_char_p()
        _lib.check(_lib.lib().pepsmg_bench_smoother(mg.h, precision, 1, 1.0, C.byref(avg), C.byref(nb), C.byref(kn)))
        assert kn.value.startswith(b"k_sweep")
        mg.destroy()
