"""Deposits of unsorted stores through cell records: the fixed-point sums, and
so every bit of rho, are those of the node grid.  A charge of 2^31 makes each
rho an integer, so a store's deposit is compared with the sum of its parts,
which are too small for records."""
import ctypes as C

import numpy as np
import pytest

from mag2d_amd import abi
from m2d_testlib import M_ION, QE, Scene, species
from test_gpu_3d import M40, Scene3
from test_gpu_bgrid import bottle

pytestmark = pytest.mark.gpu

UNIT = 2.0 ** 31
PART = 16128  # below the smallest store that uses records
FLAGS = abi.STEP_PUSH | abi.STEP_BOUNDARY | abi.STEP_DEPOSIT
DEAD = np.array([abi.DEAD_BITS], np.uint32).view(np.float32)[0]


def positions(shape, h, origin, n, rng, order):
    """Inside a grid, a tenth of the slots empty; order "cells" puts equal
    cells next to one another (sums before the atomics)."""
    p = [np.float32(o) + (rng.uniform(0, s - 1.001, n) * h).astype(np.float32) for s, o in zip(shape, origin)]
    if order == "cells":
        key = 0
        for q, s, o in zip(p, shape, origin):
            key = key * s + ((q - o) / h).astype(int)
        at = np.argsort(key, kind="stable")
        p = [q[at] for q in p]
    p[0][rng.uniform(size=n) < 0.1] = DEAD
    return p


def parts(n):
    return [slice(a, min(a + PART, n)) for a in range(0, n, PART)]


def deposit2(ctx, g, x, z):
    zero = np.zeros(len(x), np.float32)
    rho = ctx.to_device(np.zeros(g.nx * g.nz))
    abi.accumulate(ctx, g, abi.ParticlesSoA.from_host(ctx, x, z, zero, zero, zero), UNIT, rho.ptr)
    return rho.get()


@pytest.mark.parametrize("order", ["random", "cells"])
@pytest.mark.parametrize("nx,nz,n,origin", [
    (96, 96, 49151, 0.0), (96, 96, 49152, 0.0), (96, 96, 49217, -3e-3), (401, 300, 120300, 0.0),
    (401, 300, 120299, 0.0), (33, 700, 70001, 2e-3), (3, 3, 60003, 0.0), (2, 2, 49160, 0.0)])
def test_accumulate_2d(ctx, nx, nz, n, origin, order):
    h = 1e-3
    x, z = positions((nx, nz), h, (origin, origin), n, np.random.default_rng(n), order)
    g = abi.grid2d(nx, nz, h, h, origin, origin)
    want = sum(deposit2(ctx, g, x[s], z[s]) for s in parts(n))
    for _ in range(2):  # the second finds the records clear
        assert np.array_equal(deposit2(ctx, g, x, z), want)
    assert want.sum() == UNIT * (x.view(np.uint32) != abi.DEAD_BITS).sum()
    assert ctx.status(clear=True) == 0


def deposit3(ctx, g, p):
    zero = np.zeros(len(p[0]), np.float32)
    rho = ctx.to_device(np.zeros(g.nx * g.ny * g.nz))
    abi.accumulate_3d(ctx, g, abi.ParticlesSoA3D.from_host(ctx, *p, zero, zero, zero), UNIT, rho.ptr)
    return rho.get()


@pytest.mark.parametrize("order", ["random", "cells"])
@pytest.mark.parametrize("shape,n", [((17, 19, 23), 16383), ((17, 19, 23), 16384), ((17, 19, 23), 16449),
                                     ((65, 65, 65), 34327), ((65, 65, 65), 34329), ((66, 3, 130), 40001)])
def test_accumulate_3d(ctx, shape, n, order):
    h = 1e-3
    p = positions(shape, h, (0.0, 0.0, 0.0), n, np.random.default_rng(n), order)
    g = abi.grid3d(*shape, h, h, h)
    want = sum(deposit3(ctx, g, [q[s] for q in p]) for s in parts(n))
    for _ in range(2):
        assert np.array_equal(deposit3(ctx, g, p), want)
    assert ctx.status(clear=True) == 0


def test_out_of_grid_is_flagged_and_the_rest_deposited(ctx):
    g = abi.grid2d(64, 64, 1e-3, 1e-3)
    x, z = positions((64, 64), 1e-3, (0.0, 0.0), 50_000, np.random.default_rng(3), "random")
    want = deposit2(ctx, g, np.delete(x, 777), np.delete(z, 777))
    x[777], z[777] = 1.0, 0.01
    assert ctx.status(clear=True) == 0
    assert np.array_equal(deposit2(ctx, g, x, z), want)
    assert ctx.status(clear=True) == abi.FLAG_OUT_OF_RANGE


@pytest.mark.parametrize("hipos", [False, True])
@pytest.mark.parametrize("field", ["rf", "Bz", "grid"])
def test_advance_2d(ctx, field, hipos):
    """The step's own deposit, in every form of the untiled pass."""
    sc = Scene(ctx, n=128, geometry=abi.GEO_EMPTY if field == "grid" else abi.GEO_RF_22PT, rf=field == "rf",
               Bz=0.2 if field == "Bz" else 0.0, solve_oracle=field == "rf")
    if field == "grid":
        g, _, br, bz = bottle()
        sc.fields.set_magnetic_field(g, br, bz)
    rng = np.random.default_rng(5)
    n = 49_999
    x, z = positions((100, 100), sc.g.dx, (2e-3, 2e-3), n, rng, "random")
    v = [(rng.normal(size=n) * 2e4).astype(np.float32) for _ in range(3)]
    sp = species(UNIT, UNIT / QE * M_ION, 1e-9, niter=3)

    def step(s):
        P = abi.ParticlesSoA.from_host(ctx, x[s], z[s], *(c[s] for c in v), hipos=hipos)
        rho = ctx.to_device(np.zeros(128 * 128))
        abi.advance(ctx, sc.fields, sp, P, rho_ptr=rho.ptr, flags=FLAGS)
        return rho.get(), P.download()

    small = [step(s) for s in parts(n)]
    for _ in range(2):
        rho, d = step(slice(0, n))
        assert np.array_equal(rho, sum(r for r, _ in small))
        for k in d:
            assert np.array_equal(d[k], np.concatenate([e[k] for _, e in small]), equal_nan=True), k


def test_advance_3d(ctx):
    sc = Scene3(ctx)
    sc.fields.solve(1e-8)
    rng = np.random.default_rng(6)
    n = 16_450
    p = positions((30, 30, 30), sc.h, (3e-4,) * 3, n, rng, "random")
    v = [(rng.normal(size=n) * 1e3).astype(np.float32) for _ in range(3)]
    sp = abi.Species2D(UNIT, UNIT / QE * M40, 5e-9, float("inf"), 0, 0, 0)

    def step(s):
        P = abi.ParticlesSoA3D.from_host(ctx, *(c[s] for c in p + v))
        rho = ctx.to_device(np.zeros(33 ** 3))
        abi.advance_3d(ctx, sc.fields, sp, P, rho_ptr=rho.ptr, flags=FLAGS)
        return rho.get()

    want = sum(step(s) for s in parts(n))
    for _ in range(2):
        assert np.array_equal(step(slice(0, n)), want)


@pytest.mark.parametrize("axis", [0, 1])
def test_grids_longer_than_a_launch(ctx, axis):
    """Sides past the 65535 blocks (of one and of four nodes) a launch takes:
    the field's tables and the record flush on the long axis against the same
    grid with that axis along z, where a launch has room.  The weights' products
    round in another order: each within a few of their 2^31 units, and the
    step's FP32 arithmetic to 1e-5 of the kick."""
    rng = np.random.default_rng(axis)
    long, n, h = (70_000, 262_153)[axis], 300_000, 1e-4
    u = rng.normal(size=(3, 3, long))
    cells = [rng.uniform(0, 1.999, n), rng.uniform(0, 1.999, n), rng.uniform(0, long - 1.001, n)]
    out = []
    for order in ((0, 1, 2), (2, 0, 1) if axis == 0 else (0, 2, 1)):  # grid axis -> axis of u
        shape = [u.shape[a] for a in order]
        g = abi.grid3d(*shape, h, h, h)
        mask = np.full(shape, abi.FIXED, np.uint8)
        mask[1:-1, 1:-1, 1:-1] = abi.FREE
        prm = abi.Fields3DParams(g, *(h * (s - 1) for s in shape), abi.BC_FREE, 0.0, 0.0, 0.0, 1.0)
        fields = abi.Fields3D(ctx, prm, mask, np.zeros(mask.size))
        fields.upload(abi.FIELD_U, np.ascontiguousarray(u.transpose(order)))
        zero = np.zeros(n, np.float32)
        P = abi.ParticlesSoA3D.from_host(ctx, *((cells[a] * h).astype(np.float32) for a in order), zero, zero, zero)
        rho = ctx.to_device(np.zeros(mask.size))
        abi.accumulate_3d(ctx, g, P, UNIT, rho.ptr)
        sp = abi.Species2D(1.0, 1.0, 1e-9, float("inf"), 0, 0, 0)
        abi.advance_3d(ctx, fields, sp, P, flags=abi.STEP_PUSH)
        d = P.download()
        back = np.argsort(order)
        out.append((rho.get().reshape(shape).transpose(back), [d["v" + "xyz"[a]] for a in back]))
    (r0, v0), (r1, v1) = out
    assert r0.sum() == r1.sum() == UNIT * n
    assert np.abs(r0 - r1).max() <= 8 * 200  # at most 200 particles around a node, 8 units each
    for a, b in zip(v0, v1):
        assert np.abs(a - b).max() <= 1e-5 * np.abs(a).max()


def test_captured_deposit_outlives_larger_records(ctx):
    """A captured deposit replays right after a call that outgrew the records
    (it runs on the node grid)."""
    hip = C.CDLL(abi.lib()._name)  # the HIP runtime that the library itself is linked to
    g = abi.grid2d(64, 64, 1e-3, 1e-3)
    rng = np.random.default_rng(8)
    x, z = positions((64, 64), 1e-3, (0.0, 0.0), 50_000, rng, "random")
    want = deposit2(ctx, g, x, z)
    zero = np.zeros(len(x), np.float32)
    P = abi.ParticlesSoA.from_host(ctx, x, z, zero, zero, zero)
    rho = ctx.to_device(np.zeros(64 * 64))
    stream = C.c_void_p(abi.lib().m2d_ctx_stream(ctx.h))
    graph, run = C.c_void_p(), C.c_void_p()
    assert hip.hipStreamBeginCapture(stream, 1) == 0
    abi.accumulate(ctx, g, P, UNIT, rho.ptr)
    assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0
    assert hip.hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)) == 0
    big = abi.grid2d(300, 300, 1e-3, 1e-3)
    for k in range(3):
        assert hip.hipGraphLaunch(run, stream) == 0
        assert np.array_equal(rho.get(), want * (k + 1))
        xb, zb = positions((300, 300), 1e-3, (0.0, 0.0), 100_000, rng, "random")
        assert deposit2(ctx, big, xb, zb).sum() == UNIT * (xb.view(np.uint32) != abi.DEAD_BITS).sum()
    assert hip.hipGraphExecDestroy(run) == 0 and hip.hipGraphDestroy(graph) == 0
