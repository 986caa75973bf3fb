"""Batched smoothing by twos (the sweep kernel on large items, blocks on small levels): FP64 items bit for bit those
of their single-grid solves, mixed items by the residual of what they return.  The items' sizes have partial tiles on
every axis, one and two tiles along x, and one item too small for the sweeps beside four that take them; one, two and
three iterations (by blocks or one at a time, by twos, and both)."""
import pytest

from peps_mg_amd import geometry
from peps_mg_amd.batch import BatchSolver
from peps_mg_amd.multigrid import Multigrid

pytestmark = pytest.mark.gpu

DIMS = [(160, 96, 128), (40, 32, 72), (136, 104, 88), (232, 72, 64), (48, 64, 40)]   # three levels, halving
TOL = 1e-10


def sdm(d):
    return geometry.geometry_subdomain_create(geometry.geometry_domain_create(
        *d, 0.0, 0.0, 0.0, *(n / 64 for n in d), 1.01, 1.0, 1.02))


def inputs(torch, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rhs = []
    for nx, ny, nz in DIMS:
        b = torch.zeros((nz + 2, ny + 2, nx + 2), dtype=torch.float64, device="cuda")
        b[1:-1, 1:-1, 1:-1] = torch.rand((nz, ny, nx), generator=gen, device="cuda", dtype=torch.float64) * 2 - 1
        rhs.append(b)
    return rhs, [torch.zeros_like(b) for b in rhs]


@pytest.mark.parametrize("nu", [1, 2, 3])
@pytest.mark.parametrize("graph", [True, False])
def test_fp64_bitwise(nu, graph):
    import torch
    rhs, sol = inputs(torch, 31)
    B = BatchSolver([sdm(d) for d in DIMS], [3] * len(DIMS), [1] * len(DIMS), 100)
    res = B.solve_device(sol, rhs, nu, TOL, 1.0, use_graph=graph)
    torch.cuda.synchronize()
    B.destroy()
    for d, x, b, r in zip(DIMS, sol, rhs, res):
        mg = Multigrid(sdm(d), 3, 100)
        x1 = torch.zeros_like(b)
        one = mg.solve_vcycle_device(x1.data_ptr(), 0, b.data_ptr(), nu, TOL, 1.0)
        torch.cuda.synchronize()
        mg.destroy()
        assert r.cycles == one.cycles and torch.equal(x, x1), (d, r, one)


@pytest.mark.parametrize("nu", [1, 2, 3])
def test_mixed_residual(nu):
    """The residual of the returned x, from the FP64 single-grid solver started there: the same squares summed in
    another order (relative 1e-9 allowed for it)."""
    import torch
    rhs, sol = inputs(torch, 32)
    B = BatchSolver([sdm(d) for d in DIMS], [3] * len(DIMS), [1] * len(DIMS), 100, precision=1)
    first = None
    for _ in range(2):                        # a second solve from 0 replays the same schedules
        for x in sol:
            x.zero_()
        res = B.solve_device(sol, rhs, nu, TOL, 1.0)
        torch.cuda.synchronize()
        if first is None:
            first = [x.clone() for x in sol]
    B.destroy()
    for d, x, x1, b, r in zip(DIMS, sol, first, rhs, res):
        assert r.converged and r.rho < TOL and torch.equal(x, x1), (d, r)
        mg = Multigrid(sdm(d), 3, 100)
        at = mg.solve_vcycle_device(x.data_ptr(), 0, b.data_ptr(), 2, 1e30, 1.0)     # stops after one cycle
        zero = torch.zeros_like(b)
        at0 = mg.solve_vcycle_device(zero.data_ptr(), 0, b.data_ptr(), 2, 1e30, 1.0)
        torch.cuda.synchronize()
        mg.destroy()
        assert (at.res0 / at0.res0) ** 0.5 <= TOL * (1 + 1e-9), (d, at.res0, at0.res0)
