"""Records written back in record order (arrays past the Infinity Cache).

The same particles are bound once as ordinary records, which are written
back from the sorted order, and once with a 16 KB stride, which makes the
record array large enough for the other path.  Every field of every record
must come back the same, and the bytes between the records untouched.
"""
import ctypes as C

import numpy as np
import pytest

from boltzmannmfx_amd import workloads as W

pytestmark = pytest.mark.gpu

STRIDE = 16384
XPAR = [2e-5 * 50, 2e-5 * 70, 2e-5 * 30]


@pytest.mark.parametrize("segments", [False, True])
@pytest.mark.parametrize("chem", [False, True])
@pytest.mark.parametrize("steps", [0, 3])
def test_wide_records_match_ordinary_ones(bmx, gpu, segments, chem, steps):
    n = 21_003
    rng = np.random.default_rng(2)
    if segments:
        col = W.c3_hyphae(n, nroots=200, seed=4)
        mode, K, hood = bmx.NBR_STENCIL, 1, 1.1 * (4e-4 + 1e-2)
    else:
        col = W.sphere_colony(n, 0.2, 4)
        mode, K, hood = bmx.NBR_VERLET, 10, 1.0
    recs = col.recs.copy()
    recs["rdata"][:, 25:34] = rng.uniform(0.0, 2e-5, (n, 9))
    recs["idata"][:, 20:23] = rng.integers(0, 2, (n, 3))   # flags a step clears
    wide = np.full((n, STRIDE), 7, dtype=np.uint8)
    wide[:, :448] = recs.view(np.uint8).reshape(n, 448)
    ordinary = recs.copy()

    def run(bind):
        ctx = bmx.Context(0)
        ctx.set_force_params(col.fpar)
        ctx.set_geometry(col.prob_lo, col.prob_hi, col.periodic, col.n_cell)
        ctx.set_neighbor_params(mode=mode, rebuild_every=K, skin=col.skin,
                                neighborhood=hood, max_neighbors=128)
        bind(ctx)
        if segments:
            ctx.init_bonds()
        if steps:
            ctx.evolve(col.dt, steps)
        if chem:
            ctx.exchange(XPAR, 1.0)
        bmx._check(ctx.lib.bmx_sync_to_aos(ctx.h, None))
        ctx.close()

    def bind_wide(ctx):
        lay = ctx.lib.bmx_default_layout()
        lay.stride_bytes = STRIDE
        bmx._check(ctx.lib.bmx_bind_particles_aos(
            ctx.h, wide.ctypes.data_as(C.c_void_p), n, C.byref(lay), 0))
        ctx.n = n

    run(lambda ctx: ctx.bind(ordinary))
    run(bind_wide)
    # (a record's last four bytes are padding, which numpy does not copy)
    assert np.array_equal(wide[:, :444], ordinary.view(np.uint8).reshape(n, 448)[:, :444])
    assert (wide[:, 448:] == 7).all()
    if steps:
        assert not np.array_equal(ordinary["pos"], recs["pos"])
        assert not ordinary["idata"][:, 20:23].any()
