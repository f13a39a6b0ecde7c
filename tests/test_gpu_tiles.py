"""The row build and the force passes at every tile size and lane count.

A context picks its tiles (particles per wave of a force pass) and the lanes
per particle of the row build from its particle count and row length.  The
cases below reach each pair of them but segments above 60,000 (tiles of 32 at
4 and 2 lanes), with counts that leave the last tile partly empty; rows, forces, positions and (segments) integer state must equal the
oracle's bit for bit, as everywhere else.
"""
import numpy as np
import pytest

from boltzmannmfx_amd import workloads as W

pytestmark = pytest.mark.gpu


def check(ctx, st, orecs, dt, steps, segments=False):
    for k in steps:
        ctx.evolve(dt, k)
        fo = st.evolve(dt, k)
        assert np.array_equal(ctx.fc(), fo)
    off, idx = ctx.neighbors()
    ooff, oidx = st.neighbors()
    assert np.array_equal(off, ooff) and np.array_equal(idx, oidx)
    assert np.array_equal(ctx.positions(), orecs["pos"])
    if segments:
        assert np.array_equal(ctx.int_fields(), orecs["idata"])
    ctx.close()
    st.close()


# (n, phi, adhesion band, skin) and the tile and lanes per particle they get,
# the last ones with rows longer than what a tile stages on chip
SPHERES = [(1, 0.01, 6e-6, 4e-6),               # 64, 4
           (63, 0.05, 6e-6, 4e-6),
           (4097, 0.2, 6e-6, 4e-6),
           (20_011, 0.2, 6e-6, 4e-6),
           (70_001, 0.15, 6e-6, 4e-6),
           (410_003, 0.12, 6e-6, 4e-6),         # 64, 2
           (5003, 0.25, 5e-5, 5e-5),            # 8, 16
           (3001, 0.2, 5e-5, 2e-5),             # 16, 16
           (30_001, 0.25, 5e-5, 2e-5),          # 16, 8
           (61_001, 0.25, 5e-5, 2e-5),          # 16, 4
           (110_003, 0.25, 5e-5, 2e-5),         # 32, 4
           (410_011, 0.25, 5e-5, 8e-5),         # 32, 2
           (2503, 0.25, 5e-5, 1.5e-4)]          # 4, 16


@pytest.mark.parametrize("n,phi,wa,skin", SPHERES)
def test_sphere_tiles(bmx, oracle, gpu, n, phi, wa, skin):
    col = W.sphere_colony(n, phi, 5, W_A=wa, skin=skin, overlap_free=n < 50_000)
    if n == 1:  # a box of four bins
        col.prob_hi = np.array([6.2e-4, 6.2e-4, 6.2e-4])
    ctx = bmx.Context(0)
    ctx.set_force_params(col.fpar)
    ctx.set_geometry(col.prob_lo, col.prob_hi, col.periodic)
    ctx.set_neighbor_params(mode=bmx.NBR_VERLET, rebuild_every=2, skin=skin, max_neighbors=192)
    ctx.bind(col.recs.copy())
    orecs = col.recs.copy()
    g = oracle.make_geom(col.prob_lo, col.prob_hi, col.periodic, ctx.bin_dims())
    st = oracle.State(orecs, g, col.fpar, oracle.NBR_PAIR, skin, 2)
    # few steps: these overlapping inputs may exceed a period's skin / 2
    check(ctx, st, orecs, 1.0e-3 * W.DT, (1, 2))


@pytest.mark.parametrize("n", [5, 997, 25_003, 60_007])
def test_stencil_sphere_tiles(bmx, oracle, gpu, n):
    """The stencil policy's rows: tiles of 32, 4, 8 and 16 (8, 16, 8 and 4
    lanes)."""
    col = W.sphere_colony(n, 0.25, 9, W_A=5e-5, overlap_free=n < 50_000)
    hood = 1.1 * (2.0 * 7e-5 + 1e-2)
    if n == 5:
        col.prob_hi = np.array([8e-4, 8e-4, 8e-4])
    nc = [max(4, int(v // 2.0e-4)) for v in col.prob_hi]
    ctx = bmx.Context(0)
    ctx.set_force_params(col.fpar)
    ctx.set_geometry(col.prob_lo, col.prob_hi, col.periodic, nc)
    ctx.set_neighbor_params(mode=bmx.NBR_STENCIL, rebuild_every=1, neighborhood=hood,
                            max_neighbors=256)
    ctx.bind(col.recs.copy())
    orecs = col.recs.copy()
    g = oracle.make_geom(col.prob_lo, col.prob_hi, col.periodic, nc)
    st = oracle.State(orecs, g, col.fpar, oracle.NBR_STENCIL, hood, 1)
    check(ctx, st, orecs, W.DT, (1, 2))


@pytest.mark.parametrize("mode,K", [(1, 1), (0, 3)])
@pytest.mark.parametrize("n", [7, 2051, 20_483, 41_003, 50_021])
def test_segment_tiles(bmx, oracle, gpu, n, mode, K):
    """Segments: tiles of 4 (16 lanes), 8, 16 and 32 (8 lanes), either
    policy."""
    col = W.c3_hyphae(n, nroots=max(1, n // 100), seed=3)
    hood = 1.1 * (2.0 * 2.0e-4 + 1.0e-2)
    ctx = bmx.Context(0)
    ctx.set_force_params(col.fpar)
    if n == 7:
        col.prob_hi = np.array([0.04, 0.04, 0.016])
        col.n_cell = (20, 20, 8)
    ctx.set_geometry(col.prob_lo, col.prob_hi, col.periodic, col.n_cell)
    ctx.set_neighbor_params(mode=mode, rebuild_every=K, skin=col.skin, neighborhood=hood,
                            max_neighbors=384)
    ctx.bind(col.recs.copy())
    nb = ctx.bin_dims() if mode == 0 else col.n_cell
    orecs = col.recs.copy()
    g = oracle.make_geom(col.prob_lo, col.prob_hi, col.periodic, nb)
    st = oracle.State(orecs, g, col.fpar,
                      oracle.NBR_PAIR if mode == 0 else oracle.NBR_STENCIL,
                      col.skin if mode == 0 else hood, K)
    ctx.init_bonds()
    assert st.init_bonds() == 0
    check(ctx, st, orecs, col.dt, (1, 3), segments=True)


def test_colonies_in_small_tiles(bmx, gpu):
    """Two boxes in one context, tiles that straddle the colony boundary:
    each colony as it runs alone with the same bins."""
    cols = [W.sphere_colony(1003, 0.25, 1, W_A=5e-5, skin=2e-5),
            W.sphere_colony(2050, 0.2, 2, W_A=5e-5, skin=2e-5)]
    recs, starts, geoms = W.concat_colonies(cols)
    both = bmx.Context(0)
    both.set_force_params(cols[0].fpar)
    both.set_neighbor_params(mode=bmx.NBR_VERLET, rebuild_every=5, skin=2e-5)
    both.bind_colonies(recs.copy(), starts, geoms)
    both.evolve(W.DT, 12)
    got = both.positions()
    for k, col in enumerate(cols):
        one = bmx.Context(0)
        one.set_force_params(col.fpar)
        one.set_geometry(col.prob_lo, col.prob_hi, col.periodic)
        one.set_neighbor_params(mode=bmx.NBR_VERLET, rebuild_every=5, skin=2e-5)
        one.bind(col.recs.copy())
        same = one.bin_dims() == both.bin_dims(k)
        one.evolve(W.DT, 12)
        alone = one.positions()
        one.close()
        mine = got[starts[k]:starts[k + 1]]
        if same:
            assert np.array_equal(mine, alone)
        else:  # another order of the sums: 1e-16 of a force, 12 steps
            np.testing.assert_allclose(mine, alone, rtol=0, atol=1e-12 * col.prob_hi.max())
    both.close()


@pytest.mark.parametrize("first,then", [(5e-5, 6e-6), (6e-6, 5e-5)])
def test_tiles_follow_the_reach(bmx, gpu, first, then):
    """A context whose adhesion band changes after steps lays its rows out in
    the tiles of the new reach (32 and 16 here) and steps on as one bound there
    with the new band."""
    col = W.sphere_colony(24_001, 0.25, 5, W_A=5e-5, skin=2e-5, overlap_free=True)
    dt = 1.0e-3 * W.DT
    fpars = []
    for band in (first, then):
        f = np.array(col.fpar, float)
        f[0] = band
        fpars.append(f)
    def bound(fpar, recs):
        ctx = bmx.Context(0)
        ctx.set_force_params(fpar)
        ctx.set_geometry(col.prob_lo, col.prob_hi, col.periodic)
        ctx.set_neighbor_params(mode=bmx.NBR_VERLET, rebuild_every=4, skin=2e-5, max_neighbors=192)
        ctx.bind(recs)
        return ctx
    recs = col.recs.copy()
    a = bound(fpars[0], recs)
    a.evolve(dt, 5)
    a.sync()
    a.set_force_params(fpars[1])
    b = bound(fpars[1], recs.copy())
    for k in (3, 6):
        a.evolve(dt, k)
        b.evolve(dt, k)
        assert np.array_equal(a.fc(), b.fc())
        assert np.array_equal(a.positions(), b.positions())
    for x, y in zip(a.neighbors(), b.neighbors()):
        assert np.array_equal(x, y)
    a.close()
    b.close()
