"""The adjoint of the gather in the outer half cells of the grid, where its
two edges are clamped onto one: the gradient of a run that starts there
against central differences of the FP64 oracle."""
import numpy as np
import pytest

from mag2d_amd import abi
from oracle import oracle as O
from test_adjoint import M_E, QE, electrons, oracle_J, trap

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("low", [True, False])
@pytest.mark.parametrize("axis", [0, 1])
def test_gradient_of_a_run_along_an_edge(ctx, axis, low):
    n, L, N, steps, dt, Bz = 32, 2e-2, 400, 12, 1e-11, 0.1
    g, mask, volt, group, dx = trap(n, L)
    rng = np.random.default_rng(10 + axis)
    volt = volt + np.where(group >= 0, rng.uniform(-5, 5, 8)[np.maximum(group, 0)], 0.0)
    x, z, v = electrons(N, L, rng)
    v = [c * np.float32(0.1) for c in v]
    edge = (rng.uniform(0.2, 0.45, N) * dx).astype(np.float32)
    pos = [x, z]
    pos[axis] = edge if low else (np.float32(L) - edge)
    x, z = pos
    dV = (N / 1e12) / ((n - 1) ** 2)
    params = abi.FieldsParams(g, L, L, 1, 1, 0, abi.BC_FREE, 0.0, 0, 0.0, 0.0, 0.0, 0.0, Bz, 0.0, dV)
    fields = abi.Fields2D(ctx, params, mask, volt)
    P = abi.ParticlesSoA.from_host(ctx, x, z, *v)
    sp = abi.Species2D(-QE, M_E, dt, float("inf"), 0, 0, 0)
    fields.upload(abi.FIELD_U, np.zeros(n * n))
    J, grad, info = abi.adjoint_energy(ctx, fields, sp, P, steps, group=group, n_groups=8, checkpoint_every=5,
                                       adjoint_tol=1e-8)
    assert P.alive().sum() > N // 2
    og = O.grid2(n, n, dx, dx)
    p = O.particles(N)
    p["x"], p["z"], p["vx"], p["vy"], p["vz"] = x, z, *v
    h = 1e-4
    fd = np.array([(oracle_J(og, mask, volt + np.where(group == k, h, 0.0), p, dV, steps, Bz, dt) -
                    oracle_J(og, mask, volt - np.where(group == k, h, 0.0), p, dV, steps, Bz, dt)) / (2 * h)
                   for k in range(8)])
    scale = np.abs(fd).max()
    assert scale > 0
    # the bound of the run in the middle of the trap
    assert np.abs(grad - fd).max() <= 1e-4 * scale, (grad, fd)
