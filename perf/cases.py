"""What a user's program has this framework do, as cases that can be timed.

Every case is one of the programs below, at sizes and options of the
repository's own workloads, tests and decks.  Particle records live in device
memory as torch tensors (an AMReX GPU build keeps them there) and are bound in
place where the program keeps them bound; a pass returns the records' fields
after the call that writes them, or the call's own arrays.

  noalloc   one allocation-free call (bind + steps + sync) on a small colony,
            as a serving loop or a graph-capturing caller makes it
  deck      the deck driver's policy on bacteria: bins are the level mesh
            cells, the list is built every step, records synced every step
  graph     a resident colony stepped by one captured graph, then synced
  cadence   the reference's cadence, one step per call, calls enqueued without
            waiting, completed and synced every ten
  rebind    records handed over anew every step (the caller re-sorted them):
            bind, one step, sync
  segments  bonded hyphal segments in the reference's neighbour policy
  fungi     the deck driver's whole step on host records: step, division,
            exchange, fusion
  ensemble  independent colonies, each in its own box, in one graph
  adjoint   gradients of a run by the checkpointed adjoint
  coupled   a step with the particle <-> mesh coupling: volume fraction, mesh
            -> particle chemistry, amounts taken from the fluid, (segments:
            exchange,) one mechanics step, sync
"""
import ctypes
import math

import numpy as np
import torch

import boltzmannmfx_amd as bmx
from boltzmannmfx_amd import workloads

DEV = "cuda:0"
# DEM::neighborhood of the decks: 1.1 (2 r + neighbor_width)
HOOD_SPHERES = 1.1 * (2.0 * 7.0e-5 + 1.0e-2)
HOOD_SEGMENTS = 1.1 * (2.0 * 2.0e-4 + 1.0e-2)
# the fungi deck's rates: k1 k2 k3 kr1 kr2 kr3 kg kv, largest radius and length
CHEMPAR = [2.0e-5, 4.0, 2.0e-5, 2.0e-5, 6.0e-4, 2.0e-5, 4.0, 4.0e4, 2.5e-4, 35.0e-4]
XPAR = [2.0e-5, 2.0e-5, 2.0e-5]
# max_vol, max length and radius, branching and splitting probability,
# overlap, split length (the fungi deck's)
SPLIT = [6.872e-10, 35.0e-4, 2.5e-4, 0.0, 0.2, 0.2, 30.0e-4]
FUSION = [0.0, 6.0e-4, 1.0e-3, 35.0e-4]
SURFACE = 4.0e-3
CHEM_DT = 1.0e-4  # sizes stay near their start over many passes


def listed():
    return [
        # the 2,000-sphere colony in one call: launches and latency
        dict(name="noalloc_2k", kind="noalloc", n=2000, phi=0.2, skin=2.0e-5,
             wa=5.0e-5, steps=10, every=10),
        # the size of the largest shipped checkpoint, in its deck's policy
        dict(name="deck_23k", kind="deck", n=23522, phi=0.3, wa=5.0e-5, steps=1),
        # the 1,000,000-sphere colony of the benchmark
        dict(name="graph_1m", kind="graph", n=1_000_000, phi=0.3, skin=4.0e-6,
             wa=6.0e-6, steps=20, every=10),
        # an odd count at a low packing, one step per call
        dict(name="cadence_300k", kind="cadence", n=307_201, phi=0.15, skin=4.0e-6,
             wa=6.0e-6, steps=10, every=10),
        dict(name="rebind_150k", kind="rebind", n=150_000, phi=0.3, skin=4.0e-6,
             wa=6.0e-6, steps=1, every=10),
        # the 200,000-segment workload in the reference's policy
        dict(name="segments_200k", kind="segments", n=200_000, steps=10),
        # a smaller mat, ragged, records synced every step
        dict(name="segments_20k", kind="segments", n=20_011, steps=1),
        dict(name="fungi_5k", kind="fungi", n=5_003, steps=1),
        # a quarter of the 256-colony ensemble
        dict(name="ensemble_64", kind="ensemble", ncol=64, nmin=500, nmax=50_000,
             phi=0.3, skin=4.0e-6, wa=6.0e-6, steps=50, every=10),
        # the adjoint workload, checkpoints every 20 steps
        dict(name="adjoint_100k", kind="adjoint", n=100_000, phi=0.3, skin=5.0e-5,
             wa=6.0e-6, steps=40, every=10),
        # the coupling of the benchmark: about 7.6 spheres per mesh cell
        dict(name="coupled_1m", kind="coupled", n=1_000_000, segments=False, phi=0.3,
             skin=4.0e-6, wa=6.0e-6, cells=64, scheme=0),
        # segments with the trilinear scheme throughout
        dict(name="coupled_segments_100k", kind="coupled", n=100_003, segments=True,
             scheme=1),
    ]


def draw(rng):
    def count(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["noalloc", "deck", "graph", "cadence", "rebind", "segments",
                       "fungi", "ensemble", "adjoint", "coupled"])
    phi = round(rng.uniform(0.1, 0.3), 4)
    c = dict(kind=kind, phi=phi, skin=4.0e-6, wa=6.0e-6, every=10)
    if kind == "noalloc":
        return dict(c, n=count(500, 32768), steps=rng.randint(1, 20),
                    skin=rng.choice([4.0e-6, 2.0e-5]))
    if kind == "deck":
        return dict(kind=kind, n=count(500, 100_000), phi=phi, wa=5.0e-5,
                    steps=rng.randint(1, 3))
    if kind == "graph":
        return dict(c, n=count(2000, 1_000_000), steps=rng.choice([10, 20]))
    if kind == "cadence":
        return dict(c, n=count(2000, 700_000), steps=10)
    if kind == "rebind":
        return dict(c, n=count(2000, 700_000), steps=1)
    if kind == "segments":
        return dict(kind=kind, n=count(1000, 200_000), steps=rng.randint(1, 10))
    if kind == "fungi":
        return dict(kind=kind, n=count(500, 30_000), steps=1)
    if kind == "ensemble":
        return dict(c, ncol=rng.randint(2, 64), nmin=500, nmax=count(2000, 50_000),
                    steps=rng.choice([10, 20, 50]))
    if kind == "adjoint":
        return dict(c, n=count(2000, 100_000), steps=rng.choice([20, 40]), skin=5.0e-5)
    if rng.random() < 0.5:
        return dict(kind=kind, n=count(2000, 100_000), segments=True,
                    scheme=rng.randint(0, 1))
    n = count(20_000, 1_000_000)
    per_cell = rng.uniform(1.0, 16.0)
    return dict(c, n=n, segments=False, cells=max(8, int((2.0 * n / per_cell) ** (1 / 3))),
                scheme=rng.randint(0, 1))


# ------------------------------------------------------------------ inputs

def _generator(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _ints(recs):
    """The int fields of [n, 56] records: id, cpu, then idata."""
    return recs.view(torch.int32)[:, 74:111]


def _spheres(case, seed):
    """Records [n, 56] (float64 view) of a sphere colony in a 2:2:1 box,
    periodic in x and y: a randomly packed column of at most 32,768 spheres,
    repeated over x and y, radii shrunk by up to 4 per cent one by one, in
    random order."""
    n = case["n"]
    k = max(1, math.ceil(math.sqrt(n / 32768.0)))
    m = -(-n // (k * k))
    tile, lo, hi = bmx.generate_spheres(m, workloads.R_MIN, workloads.R_MAX,
                                        case["phi"], seed, (2.0 / k, 2.0 / k, 1.0))
    base = torch.from_numpy(tile.view(np.float64).reshape(m, 56)).to(DEV)
    g = _generator(seed)
    pick = torch.randperm(k * k * m, generator=g, device=DEV)[:n]
    r = base[pick % m]
    col = pick // m
    r[:, 0] += (col % k) * hi[0]
    r[:, 1] += (col // k) * hi[1]
    rad = r[:, 3] * (1.0 - 0.04 * torch.rand(n, generator=g, device=DEV, dtype=torch.float64))
    r[:, 3] = rad
    r[:, 4] = rad
    r[:, 7] = 4.0 * math.pi * rad ** 2
    r[:, 8] = 4.0 / 3.0 * math.pi * rad ** 3
    i = _ints(r)
    i[:, 0] = torch.arange(1, n + 1, device=DEV, dtype=torch.int32)
    i[:, 35] = i[:, 0]
    return r, np.zeros(3), np.array([k * hi[0], k * hi[1], hi[2]])


def _segments(case, seed):
    """A mat on a growth surface two mesh cells above the box's bottom, as
    the decks' surfaces lie inside their domains."""
    col = workloads.c3_hyphae(case["n"], nroots=max(1, case["n"] // 100), seed=seed)
    r = torch.from_numpy(col.recs.view(np.float64).reshape(-1, 56).copy()).to(DEV)
    r[:, 2] += SURFACE
    col.fpar = workloads.hyphae_fpar(z_wall=SURFACE)
    return r, col


def _species(r, seed):
    g = _generator(seed + 1)
    n = len(r)
    r[:, 28:31] = 2.0e-5 * torch.rand(n, 3, generator=g, device=DEV, dtype=torch.float64)
    r[:, 34:37] = 2.0e-12 * torch.rand(n, 3, generator=g, device=DEV,
                                       dtype=torch.float64) - 1.0e-12


def _mesh_of(case):
    """Level mesh of a coupled case."""
    if not case["segments"]:
        return (case["cells"], case["cells"], case["cells"] // 2)
    # the box of workloads.c3_hyphae
    side = math.sqrt(case["n"] * 30.0e-4 * 4.0e-4 / 0.3)
    c = max(4, int(round(side / 2.0e-3)))
    return (c, c, 8)


def _mesh_fields(n_cell, seed):
    """Species and volume fraction with one ghost layer."""
    g = _generator(seed + 2)
    nx, ny, nz = n_cell
    u = torch.rand(4, nz + 2, ny + 2, nx + 2, generator=g, device=DEV, dtype=torch.float64)
    x = torch.stack([1.0e-5 + 2.0e-5 * u[0], 1.0e-7 * u[1], 1.0e-6 + 2.0e-6 * u[2]])
    return x, 0.2 + 0.8 * u[3]


def _target(recs, seed):
    """Positions the adjoint's loss is measured from."""
    return recs[:, :3] + 1.0e-5 * torch.randn(len(recs), 3, generator=_generator(seed + 3),
                                              device=DEV, dtype=torch.float64)


def _sphere_mesh(hi):
    """Level mesh cells of 2e-4 cm, no smaller than the largest contact."""
    return tuple(max(4, int(v // 2.0e-4)) for v in hi)


def _ensemble(case, seed):
    """Colonies of sizes spread evenly over their logarithm, each in its own
    box; packings and positions by the seed."""
    rng = np.random.default_rng(seed)
    lo, hi = math.log(case["nmin"]), math.log(case["nmax"])
    sizes = np.exp(lo + (hi - lo) * (np.arange(case["ncol"]) + 0.5) / case["ncol"])
    sizes = sizes.astype(int)
    phis = rng.uniform(0.1, case["phi"], case["ncol"])
    parts, starts, geoms, boxes = [], [0], [], []
    for k, (n, phi) in enumerate(zip(sizes, phis)):
        r, blo, bhi = _spheres(dict(n=int(n), phi=float(phi)), seed * 1000 + k)
        parts.append(r)
        starts.append(starts[-1] + int(n))
        geoms.append(bmx.make_geometry(blo, bhi, (1, 1, 0)))
        boxes.append(bhi)
    return torch.cat(parts), np.array(starts, dtype=np.int64), geoms, boxes


# ----------------------------------------------------------------- programs

def _fields(recs, segments=False, chem=False):
    out = {"pos": recs[:, :3], "vel": recs[:, 9:12]}
    if segments:
        out.update(spin=recs[:, 12:15], angles=recs[:, 5:7], ints=_ints(recs))
    if chem:
        out.update(radius=recs[:, 3], length=recs[:, 4], area=recs[:, 7], vol=recs[:, 8],
                   grad=recs[:, 21:24], rates=recs[:, 24:26], species=recs[:, 28:31],
                   exchanged=recs[:, 31:34], taken=recs[:, 34:37])
    return out


def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case)
    if kind == "ensemble":
        recs, starts, geoms, _ = _ensemble(case, seed)
        torch.cuda.synchronize()
        ctx = bmx.Context(0)
        ctx.set_force_params(workloads.sphere_fpar(case["wa"]))
        ctx.set_neighbor_params(mode=bmx.NBR_VERLET, rebuild_every=case["every"],
                                skin=case["skin"], max_neighbors=64)
        lib = bmx.load_library()
        lay = lib.bmx_default_layout()
        boxes = (bmx.Geometry * len(geoms))(*geoms)
        bmx._check(lib.bmx_bind_colonies_aos(
            ctx.h, ctypes.c_void_p(recs.data_ptr()),
            starts.ctypes.data_as(ctypes.POINTER(ctypes.c_int64)), len(geoms), boxes,
            ctypes.byref(lay), bmx.AOS_DEVICE))
        ctx.n = len(recs)
        s.update(ctx=ctx, recs=recs, out=_fields(recs))
        return s
    if kind in ("segments", "fungi") or case.get("segments"):
        recs, col = _segments(case, seed)
        _species(recs, seed)
        ctx = bmx.Context(0)
        ctx.set_force_params(col.fpar)
        ctx.set_geometry(col.prob_lo, col.prob_hi, col.periodic, col.n_cell)
        ctx.set_neighbor_params(mode=bmx.NBR_STENCIL, rebuild_every=1,
                                neighborhood=HOOD_SEGMENTS, max_neighbors=256)
        if kind == "fungi":
            host = np.ascontiguousarray(recs.cpu().numpy()).view(bmx.RECORD_DTYPE).reshape(-1)
            ctx.bind(host)
            s.update(next_id=len(host) + 1, calls=0)
        else:
            torch.cuda.synchronize()
            ctx.bind_device(recs.data_ptr(), len(recs), in_place=True)
            s.update(out=_fields(recs, True, kind == "coupled"))
        ctx.init_bonds()
        s.update(ctx=ctx, recs=recs, dt=col.dt, n_cell=col.n_cell)
    else:
        recs, lo, hi = _spheres(case, seed)
        n_cell = (1, 1, 1)
        if kind == "deck":
            n_cell = _sphere_mesh(hi)
        elif kind == "coupled":
            n_cell = _mesh_of(case)
            _species(recs, seed)
        fpar = workloads.sphere_fpar(case["wa"])
        s.update(recs=recs, dt=workloads.DT, n_cell=n_cell, fpar=fpar,
                 out=_fields(recs, False, kind == "coupled"))
        torch.cuda.synchronize()
        if kind == "noalloc":
            s.update(geom=bmx.make_geometry(lo, hi, (1, 1, 0)))
            return s
        ctx = bmx.Context(0)
        ctx.set_force_params(fpar)
        ctx.set_geometry(lo, hi, (1, 1, 0), n_cell)
        if kind == "deck":
            ctx.set_neighbor_params(mode=bmx.NBR_STENCIL, rebuild_every=1,
                                    neighborhood=HOOD_SPHERES, max_neighbors=256)
        else:
            ctx.set_neighbor_params(mode=bmx.NBR_VERLET, rebuild_every=case.get("every", 10),
                                    skin=case["skin"],
                                    max_neighbors=96 if kind == "adjoint" else 64)
        if kind != "rebind":
            ctx.bind_device(recs.data_ptr(), len(recs), in_place=True)
        if kind == "adjoint":
            s.update(target=_target(recs, seed).cpu().numpy())
        s.update(ctx=ctx)
    if kind == "coupled":
        nx, ny, nz = s["n_cell"]
        x, vf = _mesh_fields(s["n_cell"], seed)
        s.update(x=x, vf=vf,
                 vf_out=torch.zeros(nz, ny, nx, device=DEV, dtype=torch.float64),
                 rhs=torch.zeros(3, nz, ny, nx, device=DEV, dtype=torch.float64))
        s["out"].update(vf=s["vf_out"], rhs=s["rhs"])
        torch.cuda.synchronize()
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "noalloc":
        bmx.evolve_aos_noalloc(s["recs"].data_ptr(), case["n"], s["geom"], s["fpar"],
                               s["dt"], case["steps"], rebuild_every=case["every"],
                               skin=case["skin"], max_neighbors=64)
        return s["out"]
    ctx = s["ctx"]
    if kind == "deck":
        for _ in range(case["steps"]):
            ctx.evolve(s["dt"], 1)
            ctx.sync()
    elif kind == "graph":
        ctx.evolve_graph(s["dt"], case["steps"])
        ctx.sync()
    elif kind == "cadence":
        for _ in range(case["steps"]):
            ctx.evolve_async(s["dt"], 1)
        ctx.wait()
        ctx.sync()
    elif kind == "rebind":
        for _ in range(case["steps"]):
            ctx.bind_device(s["recs"].data_ptr(), case["n"])
            ctx.evolve(s["dt"], 1)
            ctx.sync()
    elif kind == "segments":
        ctx.evolve(s["dt"], case["steps"])
        ctx.sync()
    elif kind == "fungi":
        s["calls"] += 1
        ctx.evolve(s["dt"], 1)
        ctx.split_particles(SPLIT, 1, s["calls"], s["next_id"])
        ctx.exchange(XPAR, s["dt"])
        recs, fused, new = ctx.fusion(FUSION, 2, s["calls"], s["next_id"])
        s["next_id"] += new
        return {"pos": recs["pos"], "real": recs["rdata"], "ints": recs["idata"]}
    elif kind == "ensemble":
        ctx.evolve_graph(workloads.DT, case["steps"])
        ctx.sync()
    elif kind == "adjoint":
        loss, g3, gr, _ = ctx.adjoint(s["dt"], case["steps"], s["target"], checkpoint_every=20)
        return {"loss": loss, "grad": g3, "grad_radius": gr}
    else:
        ctx.volume_fraction(case["scheme"], out=s["vf_out"])
        ctx.txfr_particle(CHEMPAR, s["x"], s["vf"], CHEM_DT, 4, case["scheme"],
                          case["scheme"])
        ctx.txfr_fluid(case["scheme"], out=s["rhs"])
        if case["segments"]:
            ctx.exchange(XPAR, CHEM_DT)
        ctx.evolve(s["dt"], 1)
        ctx.sync()
    return s["out"]


# Interacting or listed neighbours per particle, measured once on inputs of
# these kinds: a Verlet row at volume fraction 0.3, a segment's stencil row,
# and operations per pair as counted on the 200,000-segment workload.
ROW_SPHERE = 1.1
PAIRS_SEGMENT, FLOP_PAIR = 10.8, 476.0
FLOP_CHEM = 679.0


def work(case):
    kind = case["kind"]
    steps = case.get("steps", 1)
    if kind == "ensemble":
        lo, hi = math.log(case["nmin"]), math.log(case["nmax"])
        n = case["ncol"] * (math.exp(hi) - math.exp(lo)) / (hi - lo)
    else:
        n = case["n"]
    segments = kind in ("segments", "fungi") or bool(case.get("segments"))
    builds = -(-steps // case.get("every", 1))
    if segments:
        # position, shape, orientation and bonds read and written per step,
        # one 4-byte entry per listed pair; the state moved once per build
        step = 2 * 176.0 + 4.0 * PAIRS_SEGMENT
        build = 2 * 192.0 + 4.0 * PAIRS_SEGMENT
        flops = n * steps * PAIRS_SEGMENT * FLOP_PAIR
        synced = 24.0 + 64.0 + 140.0
    else:
        step = 68.0 + 4.0 * ROW_SPHERE
        build = 2 * 40.0 + 4.0 * ROW_SPHERE
        flops = n * steps * 60.0
        synced = 24.0 + 60.0
    total = n * (steps * step + builds * build + synced)
    if kind in ("noalloc", "rebind"):
        total += n * (40.0 + 64.0)
    if kind == "fungi":
        total += n * 2 * 448.0
    if kind == "adjoint":
        # forward, recomputed forward, and a reverse step that also reads
        # and writes the adjoint and the radius gradient
        total = n * (steps * (2 * step + step + 80.0) + 2 * builds * build + 32.0)
        flops = n * steps * 200.0
    if kind == "coupled":
        cells = math.prod(_mesh_of(case))
        total += n * (328.0 + 2 * 32.0) + 8.0 * cells * (1 + 4 + 4)
        flops += n * FLOP_CHEM
    return {"bytes": float(total), "flops": float(flops)}


# ------------------------------------------------------------ exact results

def _pairs(pos, rad, hi, reach, n_cell=None):
    """All pairs (i, j), i != j, of the +-1 cell stencil within r_i + r_j +
    reach; cells of n_cell, or no smaller than the largest such distance."""
    hi_t = torch.tensor(hi, device=DEV, dtype=torch.float64)
    if n_cell is None:
        cut = 2.0 * float(rad.max()) + reach
        n_cell = [max(1, int(v // cut)) for v in hi]
    nc = torch.tensor(n_cell, device=DEV)
    # floor(x / dx) with 1 / dx formed first, clamped to the box
    dxi = torch.tensor([1.0 / (h / c) for h, c in zip(hi, n_cell)], device=DEV,
                       dtype=torch.float64)
    c = torch.minimum(torch.floor(pos * dxi).long().clamp_(min=0), nc - 1)
    key = (c[:, 2] * nc[1] + c[:, 1]) * nc[0] + c[:, 0]
    order = torch.argsort(key)
    start = torch.searchsorted(key[order], torch.arange(int(nc.prod()) + 1, device=DEV))
    per = torch.tensor([1, 1, 0], device=DEV)
    out_i, out_j = [], []
    me = torch.arange(len(pos), device=DEV)
    seen = set()
    for off in [(x, y, z) for z in (-1, 0, 1) for y in (-1, 0, 1) for x in (-1, 0, 1)]:
        # a box of fewer than three cells along an axis meets a cell twice
        canon = tuple(o % int(nc[d]) if (d < 2 and int(nc[d]) < 3) else o
                      for d, o in enumerate(off))
        if canon in seen:
            continue
        seen.add(canon)
        q = c + torch.tensor(off, device=DEV)
        inside = ((q[:, 2] >= 0) & (q[:, 2] < nc[2]))
        q = torch.where(per.bool(), q % nc, q)
        k = (q[:, 2] * nc[1] + q[:, 1]) * nc[0] + q[:, 0]
        k = torch.where(inside, k, torch.zeros_like(k))
        a, e = start[k], torch.where(inside, start[k + 1], start[k])
        for m in range(int((e - a).max())):
            on = a + m < e
            i = me[on]
            j = order[(a + m)[on]]
            d = _image(pos[i] - pos[j], hi_t)
            near = (d.square().sum(1) <= (rad[i] + rad[j] + reach).square()) & (i != j)
            out_i.append(i[near])
            out_j.append(j[near])
    return torch.cat(out_i), torch.cat(out_j)


def _image(d, hi):
    xy = d[:, :2] - hi[:2] * torch.round(d[:, :2] / hi[:2])
    return torch.cat([xy, d[:, 2:]], 1)


def _sphere_force(pos, rad, i, j, hi, wa, mu, fpar):
    """The cubic contact law over the pairs and the growth surface."""
    d = _image(pos[i] - pos[j], hi)
    r = d.square().sum(1).sqrt()
    rs = rad[i] + rad[j]
    ra = rs + wa
    f = torch.where(r < ra, -mu * (r - ra) ** 2 * (r - rs), torch.zeros_like(r))
    a = torch.zeros_like(pos).index_add(0, i, (f / r)[:, None] * d)
    zw, wz, xi, grav = (float(fpar[k]) for k in (2, 3, 4, 5))
    dz = pos[:, 2] - zw
    rw = rad + wz
    w = torch.where(dz <= 0.0, xi * rw ** 2 * rad,
                    torch.where(dz < rw, -xi * (dz - rw) ** 2 * (dz - rad),
                                torch.zeros_like(dz)))
    w = w - grav * xi * rw ** 2 * rad
    return a + torch.stack([torch.zeros_like(w), torch.zeros_like(w), w], 1)


def _sphere_steps(pos, rad, hi, case, steps, n_cell=None):
    fpar = workloads.sphere_fpar(case["wa"])
    hi_t = torch.tensor(hi, device=DEV, dtype=torch.float64)
    vel = torch.zeros_like(pos)
    every = case.get("every", 1)
    for k in range(steps):
        if k % every == 0:
            i, j = _pairs(pos, rad, hi, case["wa"] + case.get("skin", 0.0), n_cell)
        vel = _sphere_force(pos, rad, i, j, hi_t, float(fpar[0]), float(fpar[1]), fpar)
        pos = pos + workloads.DT * vel
        pos = torch.cat([pos[:, :2] % hi_t[:2], pos[:, 2:]], 1)
    return pos, vel


def _volume_fraction(recs, hi, n_cell, scheme):
    nc = torch.tensor(n_cell, device=DEV)
    dx = torch.tensor([h / c for h, c in zip(hi, n_cell)], device=DEV, dtype=torch.float64)
    nx, ny, nz = n_cell
    # one layer below and above z for the trilinear corners outside the box
    sums = torch.zeros((nz + 2) * ny * nx, device=DEV, dtype=torch.float64)
    l = recs[:, :3] / dx + (0.5 if scheme else 0.0)
    c = torch.floor(l).long()
    f = l - c
    corners = [(x, y, z) for x in (0, 1) for y in (0, 1) for z in (0, 1)] if scheme else [(0, 0, 0)]
    for o in corners:
        q = c - (1 - torch.tensor(o, device=DEV) if scheme else 0)
        w = torch.ones(len(recs), device=DEV, dtype=torch.float64)
        if scheme:
            for d in range(3):
                w = w * (f[:, d] if o[d] else 1.0 - f[:, d])
        cell = ((q[:, 2] + 1) * ny + q[:, 1] % nc[1]) * nx + q[:, 0] % nc[0]
        sums.index_add_(0, cell, w * recs[:, 8])
    v = sums.view(nz + 2, ny, nx)[1:-1] / float(dx.prod())
    return (1.0 - v).clamp(min=0.1)


def exact(case, seed):
    """Sphere steps, their adjoint (by automatic differentiation) and the
    volume fraction.  The segment law and the chemistry have no plain
    counterpart here; their outputs are None."""
    kind = case["kind"]
    if kind == "coupled":
        if case["segments"]:
            recs, col = _segments(case, seed)
            hi, n_cell = col.prob_hi, col.n_cell
        else:
            recs, _, hi = _spheres(case, seed)
            n_cell = _mesh_of(case)
        out = dict.fromkeys(_fields(recs, case["segments"], True))
        out.update(vf=_volume_fraction(recs, hi, n_cell, case["scheme"]), rhs=None)
        return out
    if kind in ("segments", "fungi"):
        return None
    if kind == "ensemble":
        recs, starts, _, boxes = _ensemble(case, seed)
        pos, vel = [], []
        for a, b, hi in zip(starts[:-1], starts[1:], boxes):
            p, v = _sphere_steps(recs[a:b, :3], recs[a:b, 3], hi, case, case["steps"])
            pos.append(p)
            vel.append(v)
        return {"pos": torch.cat(pos), "vel": torch.cat(vel)}
    recs, _, hi = _spheres(case, seed)
    if kind != "adjoint":
        n_cell = _sphere_mesh(hi) if kind == "deck" else None
        pos, vel = _sphere_steps(recs[:, :3], recs[:, 3], hi, case, case["steps"], n_cell)
        return {"pos": pos, "vel": vel}
    target = _target(recs, seed)
    fpar = workloads.sphere_fpar(case["wa"])
    hi_t = torch.tensor(hi, device=DEV, dtype=torch.float64)
    rad = recs[:, 3].clone().requires_grad_()
    mu = torch.tensor(float(fpar[1]), device=DEV, dtype=torch.float64, requires_grad=True)
    wa = torch.tensor(float(fpar[0]), device=DEV, dtype=torch.float64, requires_grad=True)
    gamma = torch.tensor(1.0, device=DEV, dtype=torch.float64, requires_grad=True)
    pos = recs[:, :3].clone()
    i, j = _pairs(pos, recs[:, 3], hi, case["wa"] + case["skin"])
    for _ in range(case["steps"]):
        pos = pos + workloads.DT / gamma * _sphere_force(pos, rad, i, j, hi_t, wa, mu, fpar)
    loss = _image(pos - target, hi_t).square().sum() / len(pos)
    loss.backward()
    return {"loss": float(loss.detach()),
            "grad": torch.stack([mu.grad, wa.grad, gamma.grad]).cpu(),
            "grad_radius": rad.grad.cpu()}
