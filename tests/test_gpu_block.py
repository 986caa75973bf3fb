"""GPU parity of the block smoother of small levels (k_block) against the oracle: FP64 bit for bit, at the edges of
its tiles (16 x 8 x 4 and, on larger levels, 32 x 8 x 8 cells): whole tiles, one cell more or less on each axis, odd
counts, a level smaller than one tile, and stretched axes; one iteration, two in a launch, and both."""
import numpy as np
import pytest

from oracle import oracle as O
from peps_mg_amd import geometry, matrix
from peps_mg_amd.multigrid import Multigrid
from peps_mg_amd.rbgs_poisson_matrix import rbgs_iterator_fp32, rbgs_iterator_poisson_matrix

pytestmark = pytest.mark.gpu


def sdm_from(g):
    return geometry.Subdomain(g.nx, g.ny, g.nz, 0, 0, 0, g.sox, g.soy, g.soz, g.dxm, g.dym, g.dzm, g.dxg, g.dyg,
                              g.dzg, g.xg, g.yg, g.zg)


DIMS = [(16, 8, 4), (32, 16, 8), (17, 9, 5), (15, 7, 3), (2, 3, 40), (33, 31, 29),
        (96, 64, 64), (97, 65, 63), (95, 71, 49)]   # the last three: 32 x 8 x 8 tiles


@pytest.mark.parametrize("dims", DIMS)
@pytest.mark.parametrize("omega,nu", [(1.0, 1), (1.6, 2), (1.0, 5)])
def test_iterator_bitwise(dims, omega, nu):
    a = tuple(1.03 if d % 2 == 0 else 1.0 for d in dims)
    g = O.Grid(*dims, a=a)
    A = g.matrix()
    x, b = O.uniform_field(*dims, 21), O.uniform_field(*dims, 22)
    xg, x32 = x.copy(), x.astype(np.float32).astype(np.float64)
    b32, xo32 = b.astype(np.float32).astype(np.float64), x32.copy()
    rbgs_iterator_poisson_matrix(xg, matrix.MatrixHeptadiagonal(0, A), b, sdm_from(g), nu, omega)
    O.rbgs_iterator(x, A, b, nu, omega)
    assert np.array_equal(xg, x)
    # FP32 within the bound of the single-iteration kernels, 1e-6 (1 + nu) of max|x|
    rbgs_iterator_fp32(x32, b32, sdm_from(g), nu, omega)
    O.rbgs_iterator(xo32, A, b32, nu, omega)
    assert np.abs(x32 - xo32).max() <= 1e-6 * (1 + nu) * np.abs(xo32).max()


@pytest.mark.parametrize("dims,nlevel", [((48, 24, 40), 3), ((36, 20, 12), 2), ((80, 72, 64), 3), ((16, 16, 16), 2)])
@pytest.mark.parametrize("nu", [1, 2, 3])
def test_vcycle_bitwise(dims, nlevel, nu):
    """Solves on the caller's device arrays (the norm, the prolongation and the store into sol by blocks)."""
    import torch
    g = O.Grid(*dims, l=tuple(d / 16 for d in dims), a=(1.02, 1.0, 1.01))
    A = g.matrix()
    b = O.uniform_field(*dims, 23)
    mo = O.Multigrid(g, nlevel, 60)
    xo, ro = O.padded(*dims), O.padded(*dims)
    nc, hist, cit, res0 = mo.solve_vcycle(xo, ro, A, b, nu, 1e-9, 1.0)
    mg = Multigrid(sdm_from(g), nlevel, 60)
    d_b = torch.from_numpy(b).cuda()
    d_x = torch.zeros_like(d_b)
    res = mg.solve_vcycle_device(d_x.data_ptr(), 0, d_b.data_ptr(), nu, 1e-9, 1.0)
    torch.cuda.synchronize()
    assert res.cycles == nc
    assert np.max(np.abs(res.history - hist)) <= 1e-12
    assert np.array_equal(d_x.cpu().numpy(), xo)
    mg.destroy()


@pytest.mark.parametrize("dims", [(96, 80, 56), (97, 81, 57), (95, 79, 63)])
@pytest.mark.parametrize("omega,nu", [(1.0, 1), (1.6, 2), (1.0, 5)])
def test_fp32_tall_tiles(dims, omega, nu):
    """FP32 levels of 32 x 16 x 8 tiles, within the bound above."""
    g = O.Grid(*dims, a=tuple(1.03 if d % 2 == 0 else 1.0 for d in dims))   # (odd axes cannot be stretched)
    A = g.matrix()
    x = O.uniform_field(*dims, 24).astype(np.float32).astype(np.float64)
    b = O.uniform_field(*dims, 25).astype(np.float32).astype(np.float64)
    xo = x.copy()
    rbgs_iterator_fp32(x, b, sdm_from(g), nu, omega)
    O.rbgs_iterator(xo, A, b, nu, omega)
    assert np.abs(x - xo).max() <= 1e-6 * (1 + nu) * np.abs(xo).max()


@pytest.mark.parametrize("dims,nlevel", [((48, 24, 40), 3), ((144, 40, 24), 3), ((80, 72, 88), 3)])
@pytest.mark.parametrize("nu", [1, 2, 3, 4])
def test_restricting_blocks_bitwise(dims, nlevel, nu):
    """Per-level solves down to the coarsest level, whose pre-smoothing launches also restrict: partial tiles on
    every axis, the last launch of one or two iterations, from 0 and from x."""
    import torch
    g = O.Grid(*dims, l=tuple(d / 16 for d in dims), a=(1.0, 1.02, 1.01))
    A = g.matrix()
    b = O.uniform_field(*dims, 26)
    mo = O.Multigrid(g, nlevel, 4)
    xo, ro = O.padded(*dims), O.padded(*dims)
    nc, hist, cit, res0 = mo.solve_vcycle(xo, ro, A, b, nu, 1e-9, 1.0)
    mg = Multigrid(sdm_from(g), nlevel, 4, coarse_switch=0)
    d_b = torch.from_numpy(b).cuda()
    d_x = torch.zeros_like(d_b)
    res = mg.solve_vcycle_device(d_x.data_ptr(), 0, d_b.data_ptr(), nu, 1e-9, 1.0)
    torch.cuda.synchronize()
    assert res.cycles == nc
    assert np.max(np.abs(res.history - hist)) <= 1e-12
    assert np.array_equal(d_x.cpu().numpy(), xo)
