"""A tile or a look-ahead that is set selects the single-iteration smoother with it, on levels of every size; nothing
set leaves the launches of two iterations."""
import ctypes as C

import pytest

from peps_mg_amd import _lib, geometry
from peps_mg_amd.multigrid import Multigrid

pytestmark = pytest.mark.gpu


def kernel(n, precision, **opts):
    sdm = geometry.geometry_subdomain_create(geometry.geometry_domain_create(n, n, n, 0.0, 0.0, 0.0, 1.0, 1.0, 1.0))
    mg = Multigrid(sdm, 3, 1, precision=precision, **opts)
    avg, nb, kn = C.c_double(0), C.c_double(0), C.c_char_p()
    _lib.check(_lib.lib().pepsmg_bench_smoother(mg.h, precision, 1, 1.0, C.byref(avg), C.byref(nb), C.byref(kn)))
    mg.destroy()
    return kn.value.decode()


@pytest.mark.parametrize("n", [32, 64, 160])          # by blocks of both sizes and by sweeps when nothing is set
@pytest.mark.parametrize("precision,opts,tile", [
    (0, dict(tile_y=8), "<double, 64, 8, 0, 1>"), (0, dict(tile_y=16), "<double, 64, 16, 0, 1>"),
    (0, dict(tile_y=16, fused_smoother=2), "<double, 64, 16, 0, 2>"), (0, dict(fused_smoother=2), "<double, 64, 8, 0, 2>"),
    (0, dict(tile_y=32), "<double, 64, 32, 0, 1>"), (1, dict(tile_y=16), "<float, 64, 16, 0, 1>"),
    (1, dict(tile_x=64), "<float, 64, 8, 0, 1>"), (1, dict(tile_x=128, tile_y=32), "<float, 128, 32, 0, 1>"),
    (1, dict(fused_smoother=2), "<float, 64, 8, 0, 2>")])
def test_tile_set(n, precision, opts, tile):
    assert kernel(n, precision, **opts) == "k_rb_fused" + tile


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n,name", [(32, "k_block<"), (64, "k_block<"), (160, "k_sweep<")])
def test_nothing_set(n, name, precision):
    assert kernel(n, precision).startswith(name)
