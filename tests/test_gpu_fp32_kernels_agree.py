"""The FP32 smoother and prolongation kernels round alike, so a mixed-precision solve has the same values, bit for bit,
whichever of them serve its levels: single iterations in every tile and look-ahead, upward and downward, blocks of every
size with and without the prolongation and the restriction, and sweeps from x, from 0 and with the prolongation.  (The
kernels of the default route are compared with the oracle directly in the tests of sweeps and blocks.)"""
import pytest

from peps_mg_amd import geometry
from peps_mg_amd.multigrid import Multigrid

pytestmark = pytest.mark.gpu

# one level of each route: small, large and tall blocks, single iterations (3 to 4 M cells), sweeps; ragged, stretched
GRIDS = [((48, 40, 32), 3), ((72, 56, 48), 3), ((136, 104, 88), 3), ((160, 152, 144), 3), ((176, 272, 96), 4)]
TILES = [dict(tile_x=64, tile_y=8), dict(tile_x=64, tile_y=16), dict(tile_x=64, tile_y=32), dict(tile_x=128, tile_y=8),
         dict(tile_x=128, tile_y=16), dict(tile_x=128, tile_y=32), dict(tile_x=128, tile_y=16, fused_smoother=2),
         dict(tile_x=64, tile_y=8, fused_smoother=2)]


@pytest.mark.parametrize("dims,nlevel", GRIDS)
@pytest.mark.parametrize("pre,post", [(2, 2), (3, 1), (1, 4)])
def test_same_values_on_every_route(dims, nlevel, pre, post):
    import torch
    sdm = geometry.geometry_subdomain_create(geometry.geometry_domain_create(
        *dims, 0.0, 0.0, 0.0, *(n / 64 for n in dims), 1.005, 1.0, 1.01))
    nx, ny, nz = dims
    gen = torch.Generator(device="cuda").manual_seed(71)
    b = torch.zeros((nz + 2, ny + 2, nx + 2), dtype=torch.float64, device="cuda")
    b[1:-1, 1:-1, 1:-1] = torch.rand((nz, ny, nx), generator=gen, device="cuda", dtype=torch.float64) * 2 - 1
    mg = Multigrid(sdm, nlevel, 8, precision=1, inner_nu=pre, inner_nu_post=post)

    def solve(**opts):
        mg.set_options(**dict(dict(tile_x=0, tile_y=0, fused_smoother=1), **opts))
        x = torch.zeros_like(b)
        r = mg.solve_vcycle_device(x.data_ptr(), 0, b.data_ptr(), 2, 1e-10, 1.0)
        torch.cuda.synchronize()
        return x, r.rho

    x, rho = solve()
    for opts in TILES:
        xt, rt = solve(**opts)
        assert torch.equal(x, xt) and rt == rho, opts
    mg.destroy()
