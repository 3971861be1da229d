"""The direct 2D Poisson solve: fields whose free nodes fill a rectangle.

Four products with the discrete sine matrices replace the multigrid-PCG
there.  The cases sit where it can go wrong: a single free node, sides at and
past the padding (32) and the tile sizes, thin rectangles, rectangles off the
grid's centre (thick walls), the switch to the larger tiles, the largest side
and one past it (which takes the multigrid).  Each is checked against the FP64
rows of the operator, to the solve's own tolerance (1% for the reference's
rounding of the norms), and against the oracle's direct solve where that is
quick, to 1e-9 of max |u| (the residual's 1e-11 times the operator's condition
number, below 1e4 at these sizes, and a thousandth of that in practice).
"""
import ctypes as C

import numpy as np
import pytest

from mag2d_amd import abi
from oracle import oracle as O
from test_gpu_poisson_shapes import free_residual

pytestmark = pytest.mark.gpu

L, DV = 2e-2, 1e-12


def box(nx, nz, walls, seed):
    """Walls of the given thickness (x low, x high, z low, z high) at random
    voltages, random charge on the rectangle between them."""
    rng = np.random.default_rng(seed)
    a, b, c, d = walls
    mask = np.full((nx, nz), abi.FIXED, np.uint8)
    mask[a:nx - b, c:nz - d] = abi.FREE
    volt = np.where(mask == abi.FREE, 0.0, rng.normal(size=(nx, nz)) * 5)
    rho = np.where(mask == abi.FREE, rng.normal(size=(nx, nz)) * 1e-17, 0.0)
    return mask.ravel(), volt.ravel(), rho.ravel()


def fields(ctx, nx, nz, mask, volt):
    h = L / (max(nx, nz) - 1)
    g = abi.grid2d(nx, nz, h, h)
    prm = abi.FieldsParams(g, h * (nx - 1), h * (nz - 1), 0, 1, 0, abi.BC_FREE, 0.0, 0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0,
                           DV)
    return abi.Fields2D(ctx, prm, mask, volt), -(h * h) / abi.EPS0 / DV


ONE = (1, 1, 1, 1)
CASES = [(3, 3, ONE), (4, 9, ONE), (18, 18, ONE), (34, 34, ONE), (35, 66, ONE), (3, 200, ONE), (130, 5, ONE),
         (65, 97, (3, 1, 1, 7)), (128, 128, (1, 1, 2, 2)), (201, 201, ONE), (364, 387, (2, 5, 1, 1)),
         (1026, 40, ONE), (700, 1026, ONE)]


@pytest.mark.parametrize("nx,nz,walls", CASES)
def test_direct_solve_of_a_rectangle(ctx, nx, nz, walls):
    mask, volt, rho = box(nx, nz, walls, nx * 7 + nz)
    f, scale = fields(ctx, nx, nz, mask, volt)
    tol = 1e-11
    us = []
    for _ in range(2):
        f.upload(abi.FIELD_U, np.zeros(nx * nz))
        f.upload(abi.FIELD_RHO, rho)
        info = f.solve(abi.SOLVE_STATIC, tol)
        us.append(f.download(abi.FIELD_U))
    u = us[0]
    assert np.array_equal(us[0].view(np.uint64), us[1].view(np.uint64))
    assert info.rel_residual <= tol and 1 <= info.outer_iters == info.inner_iters <= 2
    pinned = mask != abi.FREE
    assert np.array_equal(u[pinned], volt[pinned])
    rn, bn = free_residual(u, mask, volt, rho, nx, nz, scale)
    assert rn <= 1.01 * tol * bn, (rn, bn)
    if nx * nz <= 20000:
        og = O.grid2(nx, nz, L / (max(nx, nz) - 1), L / (max(nx, nz) - 1))
        b = rho.copy()
        O.lib().o_poisson_rhs(C.byref(og), O.dptr(mask), O.dptr(volt), O.dptr(b), O.SOLVE_STATIC, DV)
        want = np.zeros_like(b)
        assert O.lib().o_poisson_solve(C.byref(og), O.dptr(mask), O.dptr(b), O.dptr(want)) == 0
        assert np.max(np.abs(u - want)) <= 1e-9 * np.max(np.abs(want))


def test_longer_rectangles_and_interior_electrodes_take_the_multigrid(ctx):
    mask, volt, rho = box(1027, 20, ONE, 3)
    f, scale = fields(ctx, 1027, 20, mask, volt)
    f.upload(abi.FIELD_RHO, rho)
    info = f.solve(abi.SOLVE_STATIC, 1e-10)
    assert info.inner_iters > info.outer_iters
    mask, volt, rho = box(64, 64, ONE, 4)
    mask[30 * 64 + 30] = abi.FIXED
    f, scale = fields(ctx, 64, 64, mask, volt)
    f.upload(abi.FIELD_RHO, np.where(mask == abi.FREE, rho, 0.0))
    info = f.solve(abi.SOLVE_STATIC, 1e-10)
    assert info.inner_iters > info.outer_iters and info.rel_residual <= 1e-10


def test_rf_and_raw_right_hand_sides(ctx):
    """RF: FIXED_RF walls at their voltages, FIXED ones at 0, into uRF; RAW:
    rho as it is, Dirichlet values included."""
    nx, nz = 70, 45
    mask, volt, rho = box(nx, nz, ONE, 9)
    mask[:nz] = abi.FIXED_RF
    f, scale = fields(ctx, nx, nz, mask, volt)
    f.upload(abi.FIELD_RHO, rho)
    assert f.solve(abi.SOLVE_RF, 1e-11).rel_residual <= 1e-11
    urf = f.download(abi.FIELD_URF)
    want = np.where(mask == abi.FIXED_RF, volt, 0.0)
    pinned = mask != abi.FREE
    assert np.array_equal(urf[pinned], want[pinned])
    rn, bn = free_residual(urf, mask, want, rho, nx, nz, scale)
    assert rn <= 1.01e-11 * bn
    raw = np.random.default_rng(2).normal(size=nx * nz)
    f.upload(abi.FIELD_RHO, raw)
    assert f.solve(abi.SOLVE_RAW, 1e-11).rel_residual <= 1e-11
    u = f.download(abi.FIELD_U)
    assert np.array_equal(u[pinned], raw[pinned])
    rn, bn = free_residual(u, mask, raw, raw, nx, nz, 1.0)
    assert rn <= 1.01e-11 * bn


def test_direct_solve_control(ctx):
    """A residual that is not finite adds nothing; a tolerance out of reach
    ends after 12 passes with u refined; a warm solve runs no pass."""
    nx, nz = 90, 61
    mask, volt, rho = box(nx, nz, ONE, 1)
    f, scale = fields(ctx, nx, nz, mask, volt)

    def solve(r, tol):
        f.upload(abi.FIELD_RHO, r)
        info = abi.SolveInfo()
        return abi.lib().m2d_fields2d_solve(f.h, abi.SOLVE_STATIC, tol, C.byref(info)), info

    code, info = solve(rho, 1e-30)
    assert code == -5 and info.outer_iters == 12 and info.rel_residual <= 1e-12
    code, info = solve(rho, 1e-11)
    assert code == 0 and info.outer_iters == 0
    u = f.download(abi.FIELD_U)
    bad = rho.copy()
    bad[np.flatnonzero(mask == abi.FREE)[100]] = np.nan
    code, info = solve(bad, 1e-11)
    assert code == -3 and info.outer_iters == 0
    assert np.array_equal(f.download(abi.FIELD_U), u)
