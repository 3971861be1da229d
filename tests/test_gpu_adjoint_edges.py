"""The adjoint of the gather in the outer half cells of the grid, where its
two edges are clamped onto one: the gradient of a run that starts there
against central differences of the FP64 oracle.  Stores of any slot count, the
differentiated run against the plain one, and a field that is solved,
differentiated and solved again."""
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


def small_run(ctx, n=32, L=2e-2, electrode=False):
    g, mask, volt, group, dx = trap(n, L)
    volt = volt + np.where(group >= 0, np.random.default_rng(1).uniform(-5, 5, 8)[np.maximum(group, 0)], 0.0)
    if electrode:
        mask.reshape(n, n)[3:5, 3:5] = abi.FIXED
    dV = 400 / 1e12 / (n - 1) ** 2
    params = abi.FieldsParams(g, L, L, 1, 1, 0, abi.BC_FREE, 0.0, 0, 0.0, 0.0, 0.0, 0.0, 0.1, 0.0, dV)
    return abi.Fields2D(ctx, params, mask, volt), group


def gradient(ctx, fields, group, cols, tol=0.0):
    P = abi.ParticlesSoA.from_host(ctx, *cols)
    fields.upload(abi.FIELD_U, np.zeros(group.size))
    J, grad, info = abi.adjoint_energy(ctx, fields, abi.Species2D(-QE, M_E, 1e-11, float("inf"), 0, 0, 0), P, 8,
                                       group=group, n_groups=8, checkpoint_every=3, adjoint_tol=tol)
    return J, grad, info.n_live, {k: a[P.alive()] for k, a in P.download().items()}


@pytest.mark.parametrize("count", [1, 401, 402, 403])
def test_slot_counts_of_any_remainder(ctx, count):
    """Against the same store with empty slots up to a multiple of four.  The
    gradient's atomic sums have no order; 1e-8 of it holds what that and the
    solves' 1e-10 leave."""
    fields, group = small_run(ctx)
    x, z, v = electrons(count, 2e-2, np.random.default_rng(count))
    cols = [x, z, *v]
    J, grad, live, out = gradient(ctx, fields, group, cols)
    dead = np.array([abi.DEAD_BITS], np.uint32).view(np.float32)
    pad = -count % 4
    want = gradient(ctx, fields, group, [np.concatenate([c, np.repeat(dead, pad)]) for c in cols])
    assert live == want[2] and abs(J - want[0]) <= 1e-12 * want[0]
    for k in out:
        assert np.array_equal(out[k], want[3][k]), k
    scale = np.abs(want[1]).max()
    assert scale > 0 and np.abs(grad - want[1]).max() <= 1e-8 * scale


@pytest.mark.parametrize("electrode", [False, True])
def test_the_differentiated_run_is_the_plain_run(ctx, electrode):
    """The store, u and rho end as the same steps leave them, bit for bit."""
    fields, group = small_run(ctx, electrode=electrode)
    x, z, v = electrons(1200, 2e-2, np.random.default_rng(2))
    steps, ends = 9, []
    for grad in (None, False, True):
        P = abi.ParticlesSoA.from_host(ctx, x, z, *v)
        fields.upload(abi.FIELD_U, np.zeros(group.size))
        if grad is None:
            fields.reset()
            rho = fields.ptr(abi.FIELD_RHO)
            abi.accumulate(ctx, fields.params.grid, P, -QE, rho)
            for k in range(steps):
                fields.solve(abi.SOLVE_STATIC, 1e-10)
                fields.reset()
                abi.advance(ctx, fields, abi.Species2D(-QE, M_E, 1e-11, float("inf"), k, 0, 0), P, rho_ptr=rho,
                            flags=abi.STEP_PUSH | abi.STEP_BOUNDARY | abi.STEP_DEPOSIT)
        else:
            abi.adjoint_energy(ctx, fields, abi.Species2D(-QE, M_E, 1e-11, float("inf"), 0, 0, 0), P, steps,
                               group=group if grad else None, n_groups=8, checkpoint_every=4)
        ends.append({**P.download(), "u": fields.download(abi.FIELD_U), "rho": fields.download(abi.FIELD_RHO)})
    for e in ends[1:]:
        for k in ends[0]:
            assert np.array_equal(e[k].view(np.uint8), ends[0][k].view(np.uint8)), k


@pytest.mark.parametrize("electrode", [False, True])
def test_reverse_solves_of_either_kind(ctx, electrode):
    """At the default residual a rectangle's reverse solves are the multigrid,
    at a looser one direct.  Both hold 1e-9 of a right-hand side, and at 32^2
    the operator's condition number is below 500."""
    fields, group = small_run(ctx, electrode=electrode)
    x, z, v = electrons(1200, 2e-2, np.random.default_rng(2))
    a, b = (gradient(ctx, fields, group, [x, z, *v], tol) for tol in (0.0, 1e-9))
    assert a[0] == b[0]
    assert np.abs(a[1] - b[1]).max() <= 5e-7 * np.abs(a[1]).max()


@pytest.mark.parametrize("electrode", [False, True])
def test_solves_around_a_gradient_are_the_same(ctx, electrode):
    """What a gradient or a tighter solve leaves behind may change how many
    passes the next solve queues, not what it gives: the same charge gives the
    same bits and counts before and after."""
    fields, group = small_run(ctx, electrode=electrode)
    rng = np.random.default_rng(5)
    rho = rng.normal(size=group.size) * 1e-18
    x, z, v = electrons(400, 2e-2, rng)

    def solve(tol):
        fields.upload(abi.FIELD_U, np.zeros(group.size))
        fields.upload(abi.FIELD_RHO, rho)
        info = fields.solve(abi.SOLVE_STATIC, tol)
        return info.outer_iters, info.inner_iters, info.rel_residual, fields.download(abi.FIELD_U).tobytes()

    first = solve(1e-10)
    a = gradient(ctx, fields, group, [x, z, *v])
    assert solve(1e-10) == first
    tight = solve(1e-13)
    assert solve(1e-10) == first and solve(1e-13) == tight
    b = gradient(ctx, fields, group, [x, z, *v])
    assert abs(a[0] - b[0]) <= 1e-12 * a[0] and np.abs(a[1] - b[1]).max() <= 1e-8 * np.abs(a[1]).max()


def test_a_refused_hierarchy_is_refused_alike_each_time(ctx):
    """A 4 x 850 box is solved directly, but its gradient's reverse solves, by
    multigrid, have no coarse level small enough: a bad argument, in the first
    call and in later ones, which leaves the field's own solves as they were."""
    nx, nz, h = 4, 850, 1e-4
    mask = np.full((nx, nz), abi.FIXED, np.uint8)
    mask[1:-1, 1:-1] = abi.FREE
    g = abi.grid2d(nx, nz, h, h)
    prm = abi.FieldsParams(g, h * (nx - 1), h * (nz - 1), 1, 1, 0, abi.BC_FREE, 0.0, 0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0,
                           1e-12)
    fields = abi.Fields2D(ctx, prm, mask.ravel(), np.zeros(nx * nz))
    rho = np.where(mask.ravel() == abi.FREE, np.random.default_rng(1).normal(size=nx * nz) * 1e-18, 0.0)
    P = abi.ParticlesSoA.from_host(ctx, *(np.full(4, c, np.float32) for c in (1.5e-4, 4e-2, 0.0, 0.0, 0.0)))
    us = []
    for _ in range(3):
        fields.upload(abi.FIELD_U, np.zeros(nx * nz))
        fields.upload(abi.FIELD_RHO, rho)
        assert fields.solve(abi.SOLVE_STATIC, 1e-10).rel_residual <= 1e-10
        us.append(fields.download(abi.FIELD_U).tobytes())
        with pytest.raises(abi.M2DError) as e:
            abi.adjoint_energy(ctx, fields, abi.Species2D(-QE, M_E, 1e-11, float("inf"), 0, 0, 0), P, 2,
                               group=np.full(nx * nz, -1), n_groups=1)
        assert abi.STATUS[e.value.code] == "BAD_ARG", e.value
    assert us[0] == us[1] == us[2]
