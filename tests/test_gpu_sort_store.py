"""The sort's two gathers (packed records of a scattered store, components of
a nearly ordered one), the schedule built from several blocks, and the memory
of the records."""
import ctypes as C

import numpy as np
import pytest

from mag2d_amd import abi
from m2d_testlib import M_ION, QE, Scene, species
from test_gpu_3d import Scene3

pytestmark = pytest.mark.gpu

DEAD = np.array([abi.DEAD_BITS], np.uint32).view(np.float32)[0]
FLAGS = abi.STEP_PUSH | abi.STEP_BOUNDARY | abi.STEP_DEPOSIT


def shuffled(tile, share, rng):
    """Slots in tile order, a share of them in random places."""
    order = np.argsort(tile, kind="stable")
    at = np.flatnonzero(rng.uniform(size=len(order)) < share)
    order[at] = order[rng.permutation(at)]
    return order


@pytest.mark.parametrize("hipos", [False, True])
@pytest.mark.parametrize("n,share,dead", [(1, 1.0, 0.0), (2, 1.0, 0.0), (257, 1.0, 0.2), (70_001, 0.0, 0.0),
                                          (70_001, 0.2, 0.3), (70_001, 1.0, 0.3), (262_144, 1.0, 0.1), (262_145, 0.0, 0.1),
                                          (5_000, 1.0, 1.0)])
def test_sort_2d(ctx, n, share, dead, hipos):
    sc = Scene(ctx, n=96, solve_oracle=False, geometry=abi.GEO_EMPTY, rf=False)
    rng = np.random.default_rng(n)
    pos = [rng.uniform(1e-4, sc.L * 0.999, n) for _ in range(2)]
    if not hipos:
        pos = [p.astype(np.float32).astype(np.float64) for p in pos]
    tile = abi.cell_keys(pos[0], pos[1], sc.n, sc.n, sc.g.dx, sc.g.dz) >> 6
    at = shuffled(tile, share, rng)
    pos, tile = [p[at] for p in pos], tile[at]
    v = [rng.normal(size=n).astype(np.float32) for _ in range(3)]
    gone = rng.uniform(size=n) < dead
    src = abi.ParticlesSoA.from_host(ctx, *pos, *v, hipos=hipos)
    x = src.arr["x"].get()
    x[:n][gone] = DEAD
    src.arr["x"].set(x)
    have = src.download()
    dst = abi.ParticlesSoA(ctx, n, hipos=hipos)
    live = abi.sort(ctx, sc.fields, src, dst)
    order = np.flatnonzero(~gone)[np.argsort(tile[~gone], kind="stable")]
    d = dst.download()
    assert live == len(order)
    for k in src.arr:
        assert np.array_equal(d[k][:live], have[k][order]), k
    assert (d["x"][live:].view(np.uint32) == abi.DEAD_BITS).all()


@pytest.mark.parametrize("n,share,dead", [(1, 1.0, 0.0), (40_001, 0.0, 0.2), (40_001, 1.0, 0.2), (257, 1.0, 0.5)])
def test_sort_3d(ctx, n, share, dead):
    sc = Scene3(ctx, n=33)
    rng = np.random.default_rng(n)
    pos = [rng.uniform(1e-4, sc.L * 0.999, n).astype(np.float32) for _ in range(3)]
    c = [(p.astype(np.float64) * (1.0 / sc.h)).astype(int) for p in pos]
    key = 0
    for q in c:
        key = key * 8 + q // 4
    for q in c:
        key = key * 4 + q % 4
    at = shuffled(key, share, rng)
    pos, key = [p[at] for p in pos], key[at]
    gone = rng.uniform(size=n) < dead
    pos[0][gone] = DEAD
    cols = pos + [rng.normal(size=n).astype(np.float32) for _ in range(3)]
    src, dst = abi.ParticlesSoA3D.from_host(ctx, *cols), abi.ParticlesSoA3D(ctx, n)
    live = abi.sort_3d(ctx, sc.fields, src, dst)
    order = np.flatnonzero(~gone)[np.argsort(key[~gone], kind="stable")]
    d = dst.download()
    assert live == len(order)
    for k, a in zip(abi.ParticlesSoA3D.NAMES, cols):
        assert np.array_equal(d[k][:live], a[order]), k
    assert (d["x"][live:].view(np.uint32) == abi.DEAD_BITS).all()


@pytest.mark.parametrize("n,r", [(130, 1.0), (130, 0.01), (2100, 1.0)])
def test_schedule_covers_every_particle_once(ctx, n, r):
    """The tiled pass over the schedule against the untiled pass, bit for bit:
    one block's tiles, tiles of many chunks, and more tiles (263^2) than the
    schedule's blocks have threads."""
    sc = Scene(ctx, n=n, solve_oracle=False, geometry=abi.GEO_EMPTY, rf=False)
    rng = np.random.default_rng(4)
    m = 150_000
    p = [(sc.L * (0.5 + 0.49 * r * rng.uniform(-1, 1, m))).astype(np.float32) for _ in range(2)]
    v = [(rng.normal(size=m) * 1e3).astype(np.float32) for _ in range(3)]
    a, s = abi.ParticlesSoA.from_host(ctx, *p, *v), abi.ParticlesSoA(ctx, m)
    abi.sort(ctx, sc.fields, a, s)
    c = abi.ParticlesSoA.from_host(ctx, *(s.download()[k] for k in abi.ParticlesSoA.NAMES))
    out = []
    for P in (s, c):
        rho = ctx.to_device(np.zeros(n * n))
        abi.advance(ctx, sc.fields, species(QE, M_ION, 1e-9), P, rho_ptr=rho.ptr, flags=FLAGS)
        out.append((rho.get(), P.download()))
    assert np.array_equal(out[0][0], out[1][0])
    for k in abi.ParticlesSoA.NAMES:
        assert np.array_equal(out[0][1][k].view(np.uint32), out[1][1][k].view(np.uint32)), k


def test_records_are_given_back_when_an_allocation_fails(ctx):
    """The records of sorts and deposits only make calls faster: an allocation
    that does not fit frees them before it is refused, and the next calls make
    them again."""
    hip = C.CDLL(abi.lib()._name)  # the HIP runtime that the library itself is linked to

    def free():
        ctx.sync()
        a, b = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(a), C.byref(b)) == 0
        return a.value

    sc = Scene(ctx, n=1100, solve_oracle=False, geometry=abi.GEO_EMPTY, rf=False)
    rng = np.random.default_rng(5)
    n = 2_000_000
    pos = [rng.uniform(1e-4, sc.L * 0.999, n).astype(np.float32) for _ in range(2)]
    src = abi.ParticlesSoA.from_host(ctx, *pos, *(rng.normal(size=n).astype(np.float32) for _ in range(3)))
    dst = abi.ParticlesSoA(ctx, n)
    rho = ctx.to_device(np.zeros(1100 * 1100))

    def calls():
        rho.zero()
        abi.accumulate(ctx, sc.g, src, QE, rho.ptr)
        abi.sort(ctx, sc.fields, src, dst)
        return {**dst.download(), "rho": rho.get()}

    want = calls()
    held = 32 * n + 32 * 1100 * 1100
    before = free()
    with pytest.raises(abi.M2DError) as e:
        ctx.malloc(1 << 46)
    assert abi.STATUS[e.value.code] == "NO_MEMORY"
    after = free()
    assert after - before >= held
    for _ in range(2):
        got = calls()
        for k in want:
            assert np.array_equal(got[k], want[k]), k
    assert after - free() >= held
