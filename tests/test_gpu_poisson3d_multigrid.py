"""The 3D V-cycle's own branches: two tile sizes (the large one from 2^20
nodes on), levels whose last tile is cut or whose last node lies past the fine
grid (even sides), links cut by an electrode thinner than a coarse cell, a
single dense level, a single level too large for that, a coarsest level too
large for it, swept by one workgroup or by launches (at, and one row past, the
8192 nodes a workgroup holds), and the column kernels of 4 and 8 planes.

Every solve is held to its own tolerance by the FP64 rows (1% for the
rounding of the norms), repeats bit for bit, and needs few CG iterations (a
V-cycle that mishandled a halo or a link still converges, slowly; the bound is
twice what these scenes need).
"""
import numpy as np
import pytest

from mag2d_amd import abi
from test_gpu_poisson3d_shapes import rows7, scene3

pytestmark = pytest.mark.gpu

TOL = 1e-10


def solve(ctx, shape, mask, volt, rho, most):
    nx, ny, nz = shape
    h, scale = 1e-4, 2.9e-2
    g = abi.grid3d(nx, ny, nz, h, h, h)
    prm = abi.Fields3DParams(g, h * (nx - 1), h * (ny - 1), h * (nz - 1), abi.BC_FREE, 0.0, 0.0, 0.0, scale)
    f = abi.Fields3D(ctx, prm, mask, volt)
    us = []
    for _ in range(2):
        f.upload(abi.FIELD_U, np.zeros(mask.size))
        f.upload(abi.FIELD_RHO, rho)
        info = f.solve(TOL)
        us.append(f.download(abi.FIELD_U))
    assert np.array_equal(us[0].view(np.uint64), us[1].view(np.uint64))
    assert info.rel_residual <= TOL and info.inner_iters <= most, info.inner_iters
    u, free = us[0], mask == abi.FREE
    assert np.array_equal(u[~free], volt[~free])
    b = np.where(free, -rho * scale, volt)
    A = rows7(mask, nx, ny, nz)
    beff = (b - A @ np.where(free, 0.0, b))[free]
    assert np.linalg.norm((b - A @ u)[free]) <= 1.01 * TOL * np.linalg.norm(beff)


# large tiles with cut last ones; small tiles one short of, at and past their
# sizes; even sides; a single dense level; a coarsest level swept, or thin and dense
@pytest.mark.parametrize("shape,most", [((128, 96, 90), 30), ((131, 83, 97), 30), ((101, 102, 103), 30),
                                        ((16, 33, 64), 30), ((9, 9, 9), 30), ((10, 9, 9), 30), ((5, 60, 60), 200),
                                        ((36, 36, 6), 30), ((90, 90, 6), 30), ((6, 63, 127), 30), ((6, 63, 129), 30)])
def test_levels_and_tiles(ctx, shape, most):
    mask, volt, rho = scene3(*shape, seed=sum(shape))
    solve(ctx, shape, mask, volt, rho, most)


def test_thin_grid_of_one_level(ctx):
    solve(ctx, (4, 40, 40), *scene3(4, 40, 40, seed=2), 200)


@pytest.mark.parametrize("at", [20, 21, 22, 23])
def test_thin_plates_cut_the_coarse_links(ctx, at):
    """Two plates one node thick, on and between the nodes of every coarse
    level, with a hole in one of them."""
    shape = (49, 40, 64)
    mask, volt, rho = (a.reshape(shape) for a in scene3(*shape, seed=at))
    mask[at, 4:-4, 4:-4] = abi.FIXED
    volt[at, 4:-4, 4:-4] = 3.0
    mask[8:-8, 6:-6, at + 9] = abi.FIXED
    volt[8:-8, 6:-6, at + 9] = -2.0
    mask[at, 15:20, 15:20] = abi.FREE
    volt[at, 15:20, 15:20] = 0.0
    rho = np.where(mask == abi.FREE, rho, 0.0)
    volt = np.where(mask == abi.FREE, 0.0, volt)
    solve(ctx, shape, mask.ravel(), volt.ravel(), rho.ravel(), 30)
