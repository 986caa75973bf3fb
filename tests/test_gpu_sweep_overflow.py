"""An infinity beside the faces of a level that k_sweep smooths: cells outside the level stay 0, so it spreads as the
iteration spreads it and no NaN appears (omega < 1 keeps every sum of one sign), and the cells it has not reached keep
their values."""
import numpy as np
import pytest

from oracle import oracle as O
from peps_mg_amd import geometry
from peps_mg_amd.rbgs_poisson_matrix import rbgs_iterator_fp32

pytestmark = pytest.mark.gpu

DIMS = (171, 157, 153)


@pytest.mark.parametrize("at", [(171, 157, 71), (171, 80, 72), (90, 157, 70), (1, 1, 75), (171, 157, 153), (128, 33, 60)])
@pytest.mark.parametrize("nu", [2, 4])
def test_infinity_at_the_faces(at, nu):
    g = O.Grid(*DIMS, l=tuple(float(d) for d in DIMS))
    s = geometry.Subdomain(g.nx, g.ny, g.nz, 0, 0, 0, g.sox, g.soy, g.soz, g.dxm, g.dym, g.dzm, g.dxg, g.dyg, g.dzg,
                           g.xg, g.yg, g.zg)
    x = O.uniform_field(*DIMS, 51).astype(np.float32).astype(np.float64)
    b = O.uniform_field(*DIMS, 52).astype(np.float32).astype(np.float64)
    xo = x.copy()
    O.rbgs_iterator(xo, g.matrix(), b, nu, 0.9)
    i, j, k = at
    b[k, j, i] = np.inf
    rbgs_iterator_fp32(x, b, s, nu, 0.9)
    # where the infinity is after 2 nu half-sweeps, odd i + j + k first
    z, y, w = np.ogrid[:DIMS[2] + 2, :DIMS[1] + 2, :DIMS[0] + 2]
    inside = np.zeros(x.shape, dtype=bool)
    inside[1:-1, 1:-1, 1:-1] = True
    inf = np.zeros(x.shape, dtype=bool)
    for half in range(2 * nu):
        near = inf.copy()
        for axis in range(3):
            near |= np.roll(inf, 1, axis) | np.roll(inf, -1, axis)
        near[k, j, i] = True
        inf |= near & inside & ((w + y + z) % 2 == 1 - half % 2)
    assert not np.isnan(x).any()
    assert np.array_equal(np.isinf(x), inf)
    err = np.abs(x[~inf] - xo[~inf]).max() / np.abs(xo).max()
    assert err < 1e-6 * (1 + nu), err       # the bound of the FP32 smoothers
