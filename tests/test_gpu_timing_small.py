"""The measurement hooks on levels smoothed by blocks: the launch the solver makes there, its full symbol, and the
iterations of the plain launches of a solve."""
import ctypes as C

import pytest

from peps_mg_amd import _lib, geometry
from peps_mg_amd.multigrid import Multigrid

pytestmark = pytest.mark.gpu


def solver(n, precision, nlevel=4):
    sdm = geometry.geometry_subdomain_create(geometry.geometry_domain_create(n, n, n, 0.0, 0.0, 0.0, 1.0, 1.0, 1.0))
    return Multigrid(sdm, nlevel, 60, precision=precision)


def bench_name(mg, precision):
    avg, nb, kn = C.c_double(0), C.c_double(0), C.c_char_p()
    _lib.check(_lib.lib().pepsmg_bench_smoother(mg.h, precision, 1, 1.0, C.byref(avg), C.byref(nb), C.byref(kn)))
    assert avg.value > 0
    return kn.value.decode()


@pytest.mark.parametrize("n,precision,symbol", [
    (32, 0, "k_block<double, pepsmg::BlockTile<16, 8, 4, 512>, 2, 0, false, false>"),
    (72, 0, "k_block<double, pepsmg::BlockTile<32, 8, 8, 1024>, 2, 0, false, false>"),
    (48, 1, "k_block<float, pepsmg::BlockTile<16, 8, 4, 512>, 2, 0, false, false>"),
    (64, 1, "k_block<float, pepsmg::BlockTile<32, 8, 8, 1024>, 2, 0, false, false>"),
    (80, 1, "k_block<float, pepsmg::BlockTile<32, 16, 8, 1024>, 2, 0, false, false>")])
def test_bench_names_the_launch(n, precision, symbol):
    mg = solver(n, precision, 3)
    assert bench_name(mg, precision) == symbol
    mg.destroy()


# per cycle the post-smoothing's launches from x by twos, or one by one for nu = 1 (the prolongation is a launch of its
# own on this level; pre-smoothing forms the norm, in the first cycle from the caller's arrays and then, for nu = 3, by
# two more)
@pytest.mark.parametrize("nu,nit,extra", [(1, 1, 0), (2, 2, 0), (3, 2, 2)])
def test_solve_counts_plain_iterations(nu, nit, extra):
    import torch
    mg = solver(64, 0)
    b = torch.zeros((66,) * 3, dtype=torch.float64, device="cuda")
    gen = torch.Generator(device="cuda").manual_seed(8)
    b[1:-1, 1:-1, 1:-1] = torch.rand((64,) * 3, generator=gen, device="cuda", dtype=torch.float64) * 2 - 1
    x = torch.zeros_like(b)
    L = _lib.lib()
    _lib.check(L.pepsmg_kernel_timing(mg.h, 1))
    r = mg.solve_vcycle_device(x.data_ptr(), 0, b.data_ptr(), nu, 1e-10, 1.0)
    _lib.check(L.pepsmg_kernel_timing(mg.h, 0))
    tot, cnt, name = C.c_double(0), C.c_int32(0), C.c_char_p()
    _lib.check(L.pepsmg_kernel_timing_read(mg.h, C.byref(tot), C.byref(cnt), C.byref(name)))
    assert name.value.decode() == f"k_block<double, pepsmg::BlockTile<16, 8, 4, 512>, {nit}, 0, false, false>"
    assert cnt.value == nit * r.cycles + extra and tot.value > 0
    mg.destroy()
