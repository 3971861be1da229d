"""The batched pass where a quad's lanes share trial blocks and the free-cell
answer comes a step late: segments of any length, runs of any count, slots
that start empty, ions that end on electrodes, steps across 2^32; against
each run stepped alone, bit for bit."""
import numpy as np
import pytest

from mag2d_amd import abi
from m2d_testlib import M_ION, QE, Scene
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
