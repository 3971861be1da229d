"""Collisions scattered inside the pass (a step without a deposit) against
those that a launch after the pass takes from the queue (a step with one):
the same draws from the same velocities, so the same bits.  And partners that
are part of the colliding store, which every collision reads as the push left
them."""
import numpy as np
import pytest

from mag2d_amd import abi
from m2d_testlib import M_ION, QE, Scene, ions_on_disk, species
from test_gpu_bgrid import bottle
from test_gpu_parity import _mcc_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hipos", [False, True])
@pytest.mark.parametrize("field", ["rf", "Bz", "grid"])
@pytest.mark.parametrize("n,density", [(1, 1e26), (255, 1e24), (256, 1e26), (257, 1e24), (70_001, 1e22)])
def test_pass_and_queue_agree(ctx, n, density, field, hipos):
    sc = Scene(ctx, n=96, geometry=abi.GEO_EMPTY if field == "grid" else abi.GEO_RF_22PT, rf=field == "rf",
               Bz=0.2 if field == "Bz" else 0.0, solve_oracle=field == "rf")
    if field == "grid":
        g, _, br, bz = bottle()
        sc.fields.set_magnetic_field(g, br, bz)
    dev, _ = _mcc_pair(ctx, abi.ELASTIC, density=density)
    rng = np.random.default_rng(n)
    x, z, vx, vy, vz = ions_on_disk(n, rng, r=9.9e-3, T_eV=30.0)  # some leave the box
    x[rng.uniform(size=n) < 0.1] = np.array([abi.DEAD_BITS], np.uint32).view(np.float32)[0]
    out = []
    for deposit in (False, True):
        P = abi.ParticlesSoA.from_host(ctx, x, z, vx, vy, vz, hipos=hipos)
        rho = ctx.to_device(np.zeros(sc.n * sc.n))
        flags = abi.STEP_PUSH | abi.STEP_BOUNDARY | (abi.STEP_DEPOSIT if deposit else 0)
        st = [abi.advance(ctx, sc.fields, species(QE, M_ION, 1e-9, dev.lifetime, k), P, mcc=dev,
                          rho_ptr=rho.ptr if deposit else None, flags=flags, want_stats=True) for k in range(3)]
        out.append(({k: P.arr[k].get().view(np.uint32) for k in P.arr}, [(s.collisions, s.removed) for s in st]))
    assert out[0][1] == out[1][1]
    assert n < 255 or sum(c for c, _ in out[0][1]) > 0
    for k in out[0][0]:
        assert np.array_equal(out[0][0][k], out[1][0][k]), k


@pytest.mark.parametrize("deposit", [False, True])
@pytest.mark.parametrize("part", [slice(0, None), slice(1, None), slice(500_000, None), slice(0, 300_001)])
def test_partners_from_a_part_of_the_store(ctx, part, deposit):
    """Charge exchange of ions that move alike with partners from their own
    store: whichever partner is drawn, the velocity it hands over is the one
    after the push, so all ions end with that velocity."""
    n, g = 1_000_000, abi.grid2d(64, 64, 1e-3, 1e-3)
    L = 63e-3
    mask, volt = abi.grid_build(g, abi.GEO_EMPTY, L, L)
    prm = abi.FieldsParams(g, L, L, 1, 0, 0, abi.BC_FREE, 2e3, 0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 1e-12)
    fields = abi.Fields2D(ctx, prm, mask, volt)
    rng = np.random.default_rng(3)
    x, z = ((20e-3 + 20e-3 * rng.uniform(size=n)).astype(np.float32) for _ in range(2))
    v = [np.full(n, c, np.float32) for c in (100.0, -50.0, 70.0)]
    P = abi.ParticlesSoA.from_host(ctx, x, z, *v)
    at = range(n)[part]
    partner = abi.Particles2D(*(P.arr[k].ptr + 4 * at.start for k in P.NAMES), len(at))
    mcc = abi.Mcc(ctx, M_ION, [abi.Target(M_ION, 1e24, 300.0, 0.0, partner)],
                  [abi.Interaction(abi.CX, 0, 0.0, 1e-15, 0.0, 0, 0)], 1.0)
    rho = ctx.to_device(np.zeros(64 * 64))
    flags = abi.STEP_PUSH | abi.STEP_BOUNDARY | (abi.STEP_DEPOSIT if deposit else 0)
    st = abi.advance(ctx, fields, species(QE, M_ION, 1e-9, mcc.lifetime), P, mcc=mcc,
                     rho_ptr=rho.ptr if deposit else None, flags=flags, want_stats=True)
    assert st.collisions > n // 2 and st.removed == 0
    d = P.download()
    for k, old in zip(("vx", "vy", "vz"), v):
        assert len(np.unique(d[k])) == 1, k
    assert any(d[k][0] != c[0] for k, c in zip(("vx", "vy", "vz"), v))
