"""The drop-in boundary as a caller of EvolveParticles uses it.

  * A level held as several tiles binds as one neighbour domain: the tiles'
    records step exactly as the same records bound as one array (and as the
    oracle), and rows hold pairs across tile boundaries.
  * Device records bound in place step exactly as host-bound copies, and a
    context bound once and stepped one call at a time (with a sync per call)
    steps exactly as one call of many steps.
  * bmx_refresh_from_aos: changed radii or positions re-read in place of a
    new bind give the bits of a new bind; orientation or species changes keep
    the lists.
  * bmx_evolve_async on a caller's stream, completed by bmx_wait, gives the
    bits of bmx_evolve; its errors surface at bmx_wait.
"""
import ctypes as C

import numpy as np
import pytest

from boltzmannmfx_amd import workloads as W
from conftest import HipArray

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def col():
    return W.sphere_colony(6000, 0.3, 31, W_A=6e-6, skin=4e-6)


def new_ctx(bmx, col, K=10, maxn=64):
    ctx = bmx.Context(0)
    ctx.set_force_params(col.fpar)
    ctx.set_geometry(col.prob_lo, col.prob_hi, col.periodic)
    ctx.set_neighbor_params(mode=bmx.NBR_VERLET, rebuild_every=K, skin=col.skin,
                            max_neighbors=maxn)
    return ctx


def test_tiles_bind_as_one_domain(bmx, oracle, gpu, col):
    x = col.recs["pos"][:, 0]
    L = col.prob_hi[0] - col.prob_lo[0]
    cut = col.prob_lo[0] + np.array([0.0, L / 3, 2 * L / 3, np.inf])
    tiles = [col.recs[(x >= cut[k]) & (x < cut[k + 1])].copy() for k in range(3)]
    assert all(len(t) > 0 for t in tiles)
    whole = np.concatenate(tiles).astype(bmx.RECORD_DTYPE)
    bounds = np.cumsum([0] + [len(t) for t in tiles])

    a = new_ctx(bmx, col)
    a.bind_tiles(tiles)
    a.evolve(W.DT, 25)
    off, idx = a.neighbors()
    tile_of = np.searchsorted(bounds, np.arange(len(whole)), side="right") - 1
    owner = np.repeat(np.arange(len(whole)), np.diff(off))
    assert np.any(tile_of[owner] != tile_of[idx])      # pairs across tiles
    a.sync()

    b = new_ctx(bmx, col)
    one = whole.copy()
    b.bind(one)
    b.evolve(W.DT, 25)
    b.sync()
    assert np.array_equal(np.concatenate(tiles), one)

    orecs = whole.copy()
    g = oracle.make_geom(col.prob_lo, col.prob_hi, col.periodic, b.bin_dims())
    st = oracle.State(orecs, g, col.fpar, oracle.NBR_PAIR, col.skin, 10)
    st.evolve(W.DT, 25)
    assert np.array_equal(np.concatenate(tiles)["pos"], orecs["pos"])
    a.close()
    b.close()


def test_in_place_device_records_and_per_call_cadence(bmx, gpu, col):
    ref = new_ctx(bmx, col)
    want = col.recs.copy()
    ref.bind(want)
    ref.evolve(W.DT, 23)
    ref.sync()

    d = HipArray.upload(col.recs.view(np.float64))
    try:
        ctx = new_ctx(bmx, col)
        ctx.bind_device(d.ptr.value, len(col.recs), in_place=True)
        for _ in range(23):          # EvolveParticles once per call, synced
            ctx.evolve(W.DT, 1)
            ctx.sync()
        got = np.ascontiguousarray(d.download()).view(bmx.RECORD_DTYPE).reshape(-1)
        assert np.array_equal(got, want)
        t = ctx.timing()
        assert t.steps_total == 23 and t.rebuilds_total == 3   # lists kept across calls
        ctx.close()
    finally:
        d.free()


@pytest.mark.parametrize("field", ["sizes", "positions"])
def test_refresh_equals_a_new_bind(bmx, gpu, col, field):
    ctx = new_ctx(bmx, col)
    recs = col.recs.copy()
    ctx.bind(recs)
    ctx.evolve(W.DT, 7)
    ctx.sync()
    rng = np.random.default_rng(5)
    if field == "sizes":
        recs["rdata"][:, 0] *= rng.uniform(0.97, 1.03, len(recs))
        bits = bmx.FIELD_SIZES
    else:
        recs["pos"] += rng.normal(size=recs["pos"].shape) * 1e-6
        bits = bmx.FIELD_POSITIONS
    fresh_recs = recs.copy()
    ctx.refresh(bits)
    ctx.evolve(W.DT, 15)
    fresh = new_ctx(bmx, col)
    fresh.bind(fresh_recs)
    fresh.evolve(W.DT, 15)
    assert np.array_equal(ctx.positions(), fresh.positions())
    assert np.array_equal(ctx.fc(), fresh.fc())
    ctx.close()
    fresh.close()


def test_refresh_of_other_fields_keeps_the_lists(bmx, gpu, col):
    ctx = new_ctx(bmx, col)
    recs = col.recs.copy()
    ctx.bind(recs)
    ctx.evolve(W.DT, 3)
    r0 = ctx.timing().rebuilds_total
    ctx.refresh(bmx.FIELD_ORIENTATIONS | bmx.FIELD_SPECIES)
    ctx.evolve(W.DT, 2)
    assert ctx.timing().rebuilds_total == r0
    ref = new_ctx(bmx, col)
    ref.bind(col.recs.copy())
    ref.evolve(W.DT, 5)
    assert np.array_equal(ctx.positions(), ref.positions())
    ctx.close()
    ref.close()


def hip():
    return HipArray._lib()


def test_async_on_caller_stream(bmx, gpu, col):
    s = C.c_void_p()
    assert hip().hipStreamCreate(C.byref(s)) == 0
    try:
        ctx = new_ctx(bmx, col)
        ctx.set_stream(s.value)
        ctx.bind(col.recs.copy())
        ctx.evolve_async(W.DT, 30)
        ctx.wait()
        assert ctx.query()
        ref = new_ctx(bmx, col)
        ref.bind(col.recs.copy())
        ref.evolve(W.DT, 30)
        assert np.array_equal(ctx.positions(), ref.positions())
        ctx.set_stream(0)
        ctx.evolve_async(W.DT, 5)
        ref.evolve(W.DT, 5)
        assert np.array_equal(ctx.positions(), ref.positions())  # completes first
        ctx.close()
        ref.close()
        # an overflow of asynchronous steps is reported by the wait
        bad = new_ctx(bmx, col, maxn=1)
        bad.bind(col.recs.copy())
        bad.evolve_async(W.DT, 2)
        with pytest.raises(bmx.BMXError) as e:
            bad.wait()
        assert e.value.code == 5
        bad.close()
    finally:
        hip().hipStreamDestroy(s)


def test_chained_async_calls(bmx, gpu, col):
    """One step per call, enqueued back to back without waiting, completed
    by one wait: the bits of one call of as many steps."""
    ctx = new_ctx(bmx, col)
    ctx.bind(col.recs.copy())
    for _ in range(25):
        ctx.evolve_async(W.DT, 1)
    ctx.wait()
    ref = new_ctx(bmx, col)
    ref.bind(col.recs.copy())
    ref.evolve(W.DT, 25)
    assert np.array_equal(ctx.positions(), ref.positions())
    assert ctx.timing().rebuilds_total == 3
    ctx.close()
    ref.close()


def test_fc_survives_reorders_after_the_step(bmx, oracle, gpu):
    """The forces of the last step, and the velocities a sync writes from
    them, are the same whether they are read at once or after passes that
    reorder the particles (one exchange, several, bond detection)."""
    rng = np.random.default_rng(12)
    for segments in (True, False):
        col = (W.c3_hyphae(2003, nroots=20, seed=3) if segments
               else W.sphere_colony(3001, 0.25, 3, skin=2e-5))
        n = len(col.recs)
        col.recs["rdata"][:, 5] = 1e-12
        col.recs["rdata"][:, 25:28] = rng.uniform(0, 2e-5, (n, 3))
        ctx = bmx.Context(0)
        ctx.set_force_params(col.fpar)
        ctx.set_geometry(col.prob_lo, col.prob_hi, col.periodic, col.n_cell)
        if segments:
            ctx.set_neighbor_params(mode=bmx.NBR_STENCIL, rebuild_every=1,
                                    neighborhood=1.1 * (4e-4 + 1e-2), max_neighbors=256)
        else:
            ctx.set_neighbor_params(mode=bmx.NBR_VERLET, rebuild_every=10, skin=col.skin)
        recs = col.recs.copy()
        ctx.bind(recs)
        ctx.evolve((100 if segments else 1) * col.dt, 3)
        fc = ctx.fc()
        ctx.sync()
        vel = recs["rdata"][:, 6:12].copy()
        assert np.abs(fc[:3]).max() > 0 and np.array_equal(vel, fc.T)
        passes = [lambda: ctx.exchange([0.0] * 3, 1.0)] * 3
        passes.append(ctx.init_bonds)
        for k, call in enumerate(passes):
            call()
            assert np.array_equal(ctx.fc(), fc), k
        recs["rdata"][:, 6:12] = 0.0
        ctx.exchange([0.0] * 3, 1.0)
        ctx.sync()
        assert np.array_equal(recs["rdata"][:, 6:12], vel)
        ctx.evolve(col.dt, 1)
        assert not np.array_equal(ctx.fc(), fc)
        ctx.close()


def test_fc_of_the_call_before_a_failed_guarded_call(bmx, gpu):
    """A guarded call that ends in its first period (a row over the capacity)
    has not reached the step that writes the forces: those of the call before
    are still there, in their particles' order."""
    col = W.sphere_colony(3001, 0.25, 3, skin=2e-5)
    ctx = bmx.Context(0)
    ctx.set_force_params(col.fpar)
    ctx.set_geometry(col.prob_lo, col.prob_hi, col.periodic, col.n_cell)
    ctx.set_neighbor_params(mode=bmx.NBR_VERLET, rebuild_every=10, skin=col.skin,
                            max_neighbors=24)
    ctx.set_guard(True)
    recs = col.recs.copy()
    ctx.bind(recs)
    dt = 1e-9 * col.dt
    ctx.evolve(dt, 25)
    fc = ctx.fc()
    rng = np.random.default_rng(5)
    recs["pos"] = recs["pos"][rng.permutation(len(recs))]
    mid = 0.5 * (np.asarray(col.prob_lo) + np.asarray(col.prob_hi))
    recs["pos"][:40] = mid + rng.uniform(-1e-5, 1e-5, (40, 3))
    ctx.refresh(bmx.FIELD_POSITIONS, recs)
    with pytest.raises(bmx.BMXError) as e:
        ctx.evolve(dt, 45)
    assert e.value.code == 5                          # a row over the capacity
    assert np.array_equal(ctx.fc(), fc)
    ctx.close()


@pytest.mark.parametrize("nsteps", [7, 13, 20])
def test_fc_of_a_guarded_call_that_fails_in_its_last_two_periods(bmx, gpu, nsteps):
    """Two periods are in flight, so a guarded call that fails (a row over the
    capacity) in one of its last two has taken the step that writes the
    forces: those of the same steps without the guard, which fail alike."""
    col = W.sphere_colony(3001, 0.25, 3, skin=2e-5)
    rng = np.random.default_rng(5)
    mid = 0.5 * (np.asarray(col.prob_lo) + np.asarray(col.prob_hi))
    moved = col.recs["pos"][rng.permutation(len(col.recs))].copy()
    moved[:40] = mid + rng.uniform(-1e-5, 1e-5, (40, 3))
    dt = 1e-9 * col.dt
    got = []
    for guard in (False, True):
        ctx = new_ctx(bmx, col, maxn=24)
        ctx.set_guard(guard)
        recs = col.recs.copy()
        ctx.bind(recs)
        ctx.evolve(dt, 25)
        recs["pos"] = moved
        ctx.refresh(bmx.FIELD_POSITIONS, recs)
        with pytest.raises(bmx.BMXError) as e:
            ctx.evolve(dt, nsteps)
        assert e.value.code == 5                      # a row over the capacity
        fc, pos = ctx.fc(), ctx.positions()
        ctx.sync()
        assert np.array_equal(recs["rdata"][:, 6:12], fc.T)
        got.append((fc, pos))
        ctx.close()
    assert np.abs(got[0][0][:3]).max() > 0
    for a, b in zip(*got):
        assert np.array_equal(a, b)
