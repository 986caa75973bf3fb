"""CG iterations on levels with many blocks: those whose partial sums one block adds up between the kernels, and those
whose march has more blocks than there is room for partial sums, which run the separate mat-vec, dot product and
direction update."""
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


@pytest.mark.parametrize("ny", [1100000, 4300000])
def test_start_from_zero(ny):
    """One inner cycle of a mixed solve, whose finest level starts from x = 0, is the oracle's first CG(4) V-cycle
    from x = 0 but for its rounding: nine CG steps' worth of the FP32 smoothers' bound, 1e-6 each, for the
    solution (relative to its maximum) and for the residual (relative to the right-hand side: on a level two cells
    wide and deep, whose matrix has a condition number below 10, it shares the solution's relative error)."""
    dims = (2, ny, 2)
    g = O.Grid(*dims, l=tuple(float(d) for d in dims))
    b = O.uniform_field(*dims, 44)
    mo = O.Multigrid(g, 2, 1, smoother=1)
    xo, ro = O.padded(*dims), O.padded(*dims)
    _, hist, _, _ = mo.solve_vcycle(xo, ro, g.matrix(), b, 4, 1e-12, 1.0)
    mg = Multigrid(sdm_from(g), 2, 1, smoother=1, precision=1, inner_cycles=1, inner_nu=4, inner_nu_post=4)
    x, r = O.padded(*dims), O.padded(*dims)
    res = mg.solve_vcycle(x, r, None, b, 4, 1e-12, 1.0)
    mg.destroy()
    assert res.cycles == 1
    assert np.abs(x - xo).max() <= 9e-6 * np.abs(xo).max()
    assert abs(res.rho - hist[0]) <= 9e-5, (res.rho, hist[0])


@pytest.mark.parametrize("dims", [(2, 65000, 2), (2, 65600, 2), (3, 140000, 2)])
@pytest.mark.parametrize("nu", [1, 4])
def test_iterator_from_x(dims, nu):
    """At and beyond the count of partial sums (4096) up to which every block adds them up itself.  The sums of at
    most 840000 products are ordered differently: about 1e-13 relative each (the square root of their number times
    the rounding unit), carried through four iterations of a well-conditioned system; bounds 100 times that."""
    g = O.Grid(*dims, l=tuple(float(d) for d in dims))
    A = g.matrix()
    x, b = O.uniform_field(*dims, 45), O.uniform_field(*dims, 46)
    xg = x.copy()
    cg_iterator_poisson_matrix(xg, None, b, sdm_from(g), nu)
    O.cg_iterator(x, A, b, nu)
    np.testing.assert_allclose(xg, x, rtol=1e-11, atol=1e-11 * np.abs(x).max())
