"""The batched pass where a quad's lanes share trial blocks and the free-cell
answer comes a step late: segments of any length, runs of any count, slots
that start empty, ions that end on electrodes, steps across 2^32; and every
form of the pass in a box wider than its grid; against each run stepped
alone, bit for bit."""
import numpy as np
import pytest

from mag2d_amd import abi
from m2d_testlib import M_HE, M_ION, QE, Scene
from test_batch import _runs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ppt,block", [(1, 64), (2, 128), (4, 256)])
@pytest.mark.parametrize("seg,steps,first", [(1, 3, 0), (3, 8, 1), (5, 5, 2 ** 32 - 3), (64, 41, 7)])
def test_segments(ctx, seg, steps, first, ppt, block):
    sc = Scene(ctx, n=64)
    rng = np.random.default_rng(seg)
    counts, dens = [1, 0, 6, 255, 1027, 2], [1e24, None, 1e23, 1e22, 3e23, 1e24]
    stores, mccs = _runs(ctx, sc, counts, [20.0] * 6, dens, rng)
    for s in stores:  # hot: some leave, some hit an electrode, some slots are empty
        for v in s[2:]:
            v *= np.float32(30.0)
        if len(s[0]) > 10:
            s[0][::11] = np.array([abi.DEAD_BITS], np.uint32).view(np.float32)[0]
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int64)
    B = abi.ParticlesSoA.from_host(ctx, *[np.concatenate([s[c] for s in stores]) for c in range(5)])
    amps = [5.0, 1.0, 30.0, 60.0, 12.0, 44.0]
    batch = abi.Batch(ctx, sc.fields, abi.Species2D(QE, M_ION, 1e-9, float("inf"), 0, 0, 0), B, offsets, amps, mccs)
    batch.set_shape(block, ppt, seg)
    batch.advance(first, steps)
    got = {k: a.get() for k, a in B.arr.items()}
    for r, n in enumerate(counts):
        if n == 0:
            continue
        P = abi.ParticlesSoA.from_host(ctx, *stores[r])
        fr = abi.Fields2D(ctx, abi.FieldsParams(sc.g, sc.L, sc.L, 0, 0, 0, abi.BC_FREE, 0.0, 1, amps[r],
                                                sc.params.rf_omega, 0.0, 0.0, 0.0, 0.0, sc.dV), sc.mask, sc.volt)
        fr.upload(abi.FIELD_U, sc.u)
        fr.upload(abi.FIELD_URF, sc.urf)
        for k in range(steps):
            abi.advance(ctx, fr, abi.Species2D(QE, M_ION, 1e-9, mccs[r].lifetime, first + k, r, 0), P, mcc=mccs[r])
        alive, d = P.alive(), P.download()
        here = slice(offsets[r], offsets[r + 1])
        assert np.array_equal(alive, got["x"][here].view(np.uint32) != abi.DEAD_BITS), r
        for c in abi.ParticlesSoA.NAMES:
            assert np.array_equal(d[c][alive].view(np.uint32), got[c][here][alive].view(np.uint32)), (r, c)


@pytest.mark.parametrize("ppt", [1, 2, 4])
@pytest.mark.parametrize("hipos", [False, True])
@pytest.mark.parametrize("form", ["specialised", "Bz", "origin", "periodic"])
def test_box_wider_than_its_grid(ctx, form, hipos, ppt):
    """Ions that end in the last row of nodes, up to 0.9 cells past the last
    node, are removed there and look up no field afterwards: past half a cell
    that look-up would raise the out-of-range flag, which no run stepped alone
    raises."""
    n, h, steps = 48, 1e-3, 12
    o = -3e-3 if form == "origin" else 0.0
    end = o + (n - 1 + 0.9) * h
    g = abi.grid2d(n, n, h, h, o, o)
    mask, volt = abi.grid_build(abi.grid2d(n, n, h, h), abi.GEO_EMPTY, (n - 1) * h, (n - 1) * h)
    mask.reshape(n, n)[20:24, 20:24] = abi.FIXED
    prm = [abi.FieldsParams(g, end, end, 0, 0, 0, abi.BC_PERIODIC if form == "periodic" else abi.BC_FREE, 0.0, 1, amp,
                            1e8, 0.0, 0.0, 0.05 if form == "Bz" else 0.0, 0.0, 1e-12) for amp in (5.0, 20.0, 40.0)]
    rng = np.random.default_rng(8)
    u = rng.normal(size=(2, n * n))
    fields = [abi.Fields2D(ctx, p, mask, volt) for p in prm]
    for f in fields:
        f.upload(abi.FIELD_U, u[0])
        f.upload(abi.FIELD_URF, u[1])
    counts = [203, 5, 310]
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int64)
    N = int(offsets[-1])
    # two rows inside the last nodes on either axis, up to 1.3 cells a step
    pos = [o + h * rng.uniform(2.0, n - 1.5, N) for _ in range(2)]
    near = rng.uniform(size=N) < 0.5
    pos[0][near], pos[1][~near] = [o + h * rng.uniform(n - 4.0, n - 1.5, m.sum()) for m in (near, ~near)]
    dt = 1e-9
    v = [(rng.uniform(-1.3, 1.3, N) * h / dt).astype(np.float32) for _ in range(3)]
    if not hipos:
        pos = [p.astype(np.float32) for p in pos]
    gas = abi.Mcc(ctx, M_ION, [abi.Target(M_HE, 1e22, 300.0, 0.0, abi.Particles2D())],
                  [abi.Interaction(abi.ELASTIC, 0, 0.0, 1e-15, 0.0, 0, 0)], 1.0)
    mccs = [None, gas, gas]
    ctx.status(clear=True)
    runs = []
    for r in range(3):
        here = slice(offsets[r], offsets[r + 1])
        P = abi.ParticlesSoA.from_host(ctx, *(c[here] for c in pos + v), hipos=hipos)
        life = mccs[r].lifetime if mccs[r] else float("inf")
        for k in range(steps):
            abi.advance(ctx, fields[r], abi.Species2D(QE, M_ION, dt, life, k, r, 0), P, mcc=mccs[r])
        runs.append((P.alive(), P.download()))
    assert ctx.status(clear=True) == 0
    assert 0 < sum((~a).sum() for a, _ in runs) < N
    B = abi.ParticlesSoA.from_host(ctx, *pos, *v, hipos=hipos)
    batch = abi.Batch(ctx, fields[0], abi.Species2D(QE, M_ION, dt, float("inf"), 0, 0, 0), B, offsets,
                      [5.0, 20.0, 40.0], mccs)
    batch.set_shape(64, ppt, 5)
    batch.advance(0, steps)
    assert ctx.status(clear=True) == 0
    got = {k: a.get() for k, a in B.arr.items()}
    for r, (alive, d) in enumerate(runs):
        here = slice(offsets[r], offsets[r + 1])
        assert np.array_equal(alive, got["x"][here].view(np.uint32) != abi.DEAD_BITS), r
        for c in B.arr:
            assert np.array_equal(d[c][alive].view(np.uint32), got[c][here][alive].view(np.uint32)), (r, c)
