"""CG iterations on levels that one workgroup holds (up to 2048 pairs of cells along x) against the oracle: the
smallest, partial and full counts of pairs per thread, odd rows, and a level beyond the limit.  The sums of the dot
products are ordered differently, so values agree to rounding (bounds as for the separate kernels)."""
import numpy as np
import pytest

from oracle import oracle as O
from peps_mg_amd import geometry
from peps_mg_amd.cg_poisson_matrix import cg_iterator_poisson_matrix
from peps_mg_amd.multigrid import Multigrid

pytestmark = pytest.mark.gpu


def sdm_from(g):
    return geometry.Subdomain(g.nx, g.ny, g.nz, 0, 0, 0, g.sox, g.soy, g.soz, g.dxm, g.dym, g.dzm, g.dxg, g.dyg,
                              g.dzg, g.xg, g.yg, g.zg)


@pytest.mark.parametrize("dims", [(2, 2, 2), (3, 5, 7), (8, 8, 8), (16, 16, 8), (17, 11, 10), (16, 16, 16),
                                  (64, 8, 8), (2, 32, 64), (66, 8, 8)])
@pytest.mark.parametrize("nu", [1, 2, 6])
def test_iterator(dims, nu):
    g = O.Grid(*dims, a=tuple(1.03 if d % 2 == 0 else 1.0 for d in dims))
    A = g.matrix()
    x, b = O.uniform_field(*dims, 41), O.uniform_field(*dims, 42)
    xg = x.copy()
    cg_iterator_poisson_matrix(xg, None, b, sdm_from(g), nu)
    O.cg_iterator(x, A, b, nu)
    np.testing.assert_allclose(xg, x, rtol=1e-11, atol=1e-12 * np.abs(x).max())


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("dims", [(32, 32, 32), (40, 24, 16)])
def test_solve(dims, precision):
    """CG(4) V-cycles: the residual of the returned x, from the red/black FP64 solver started there (1e-9 relative
    for the order of its sum)."""
    import torch
    g = O.Grid(*dims, l=tuple(d / 32 for d in dims))
    b = torch.from_numpy(O.uniform_field(*dims, 43)).cuda()
    x = torch.zeros_like(b)
    mg = Multigrid(sdm_from(g), 3, 100, smoother=1, precision=precision)
    res = mg.solve_vcycle_device(x.data_ptr(), 0, b.data_ptr(), 4, 1e-10, 1.0)
    rb = Multigrid(sdm_from(g), 3, 100)
    zero = torch.zeros_like(b)
    at = rb.solve_vcycle_device(x.data_ptr(), 0, b.data_ptr(), 2, 1e30, 1.0)
    at0 = rb.solve_vcycle_device(zero.data_ptr(), 0, b.data_ptr(), 2, 1e30, 1.0)
    torch.cuda.synchronize()
    assert res.converged
    assert (at.res0 / at0.res0) ** 0.5 <= 1e-10 * (1 + 1e-9)
