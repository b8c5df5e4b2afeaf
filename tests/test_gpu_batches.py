"""What may not depend on how a job is cut into launches: the fields, the
frames that an engine accepts, and its memory."""
import numpy as np
import pytest

from pyglasstools_amd import engine, workload

pytestmark = pytest.mark.gpu
RMAX = 1.25 * 1.62


def _stack(frames, key):
    import torch

    return torch.tensor(np.stack([f[key] for f in frames]), dtype=torch.float64, device="cuda")


def _fields(e, frames, fields, first=0, count=None, per_launch=None):
    """Fields of frames first .. first + count - 1 as one job."""
    import torch

    sel = frames[first:first + (count or len(frames))]
    if per_launch:
        e.set_tuning(frames_per_launch=per_launch)
    out = {k: torch.full((len(sel), e.G, e.dim, e.dim), np.nan, dtype=torch.float64, device="cuda") for k in fields}
    pos, diam, mass, vel = (_stack(sel, k) for k in ("pos", "diam", "mass", "vel"))
    disp = _stack(sel, "disp") if "elastic" in fields else None
    torch.cuda.synchronize()
    e.compute_frames(len(sel), len(sel[0]["diam"]), pos, diam, mass, vel, disp, fields=fields,
                     **{"d_" + k: v for k, v in out.items()})
    torch.cuda.synchronize()
    return {k: v.cpu().numpy() for k, v in out.items()}


def _frames(dim, N, nf, seed):
    frames = [workload.make_system(N, dim, seed + f) for f in range(nf)]
    rng = np.random.default_rng(seed)
    for s in frames:
        s["disp"] = rng.normal(0.0, 0.02, (N, 3)) * np.array([1, 1, 1 if dim == 3 else 0])
    return frames


def _grid(kind, L, dim, side):
    if kind == "scattered":
        return np.random.default_rng(3).uniform(-0.6 * L, 0.6 * L, (side ** dim, 3)) * np.array([1, 1, float(dim == 3)])
    return workload.cartesian_grid_2d(L, side) if dim == 2 else workload.cartesian_grid_3d(L, side)


@pytest.mark.parametrize("dim,N,side,nf,fields,prec,kind,periodic", [
    (2, 2000, 32, 200, ("virial", "kinetic"), "fp64", "lattice", None),
    (2, 2000, 32, 200, ("virial", "kinetic"), "fp32", "lattice", None),
    (2, 6200, 32, 200, ("virial", "elastic"), "fp64", "lattice", None),
    (2, 9000, 64, 50, ("virial",), "fp64", "lattice", (0, 1, 0)),
    (2, 1500, 40, 140, ("virial", "kinetic"), "fp64", "scattered", None),
    (2, 500, 8, 3100, ("virial", "kinetic"), "fp64", "lattice", None),
    (3, 4000, 12, 120, ("virial", "kinetic"), "fp64", "lattice", None),
    (3, 4000, 12, 120, ("virial",), "fp32", "lattice", None),
    (3, 3000, 16, 50, ("virial", "kinetic", "elastic"), "fp64", "scattered", None)])
def test_fields_do_not_depend_on_the_launch(gpu, dim, N, side, nf, fields, prec, kind, periodic):
    """A job of many frames takes whole tiles of the grid, one of a few frames
    parts of them.  Windows of more particles than a tile's list holds (128),
    one to four lists' worth: the same fields bit for bit, all frames in a
    launch, 24 of them (half or quarter tiles) and one by one."""
    print("launches %dD N=%d side %d x %d %s %s %s" % (dim, N, side, nf, fields, prec, kind), flush=True)
    frames = _frames(dim, N, min(nf, 24), 12000)
    many = [frames[k % len(frames)] for k in range(nf)]
    e = engine.Engine(dim=dim, max_rcut=RMAX, precision=prec)
    e.set_box(frames[0]["L"], frames[0]["periodic"] if periodic is None else periodic)
    e.set_grid(_grid(kind, frames[0]["L"][0], dim, side))
    whole = _fields(e, many, fields, per_launch=nf)
    some = _fields(e, frames, fields, per_launch=24)
    for k in fields:
        assert np.isfinite(whole[k]).all() and np.abs(whole[k]).max() > 0
        for f in range(nf):
            assert np.array_equal(whole[k][f], some[k][f % len(frames)]), (k, f)
    for f in (0, 13):
        one = _fields(e, frames, fields, first=f, count=1)
        for k in fields:
            assert np.array_equal(whole[k][f], one[k][0]), (k, f)


@pytest.mark.parametrize("dim,spec", [(2, ((2000, 1, 32), (6200, 2, 32), (9000, 1, 40), (500, 30, 30))),
                                      (3, ((4000, 1, 12), (3000, 3, 9), (9000, 20, 20)))])
def test_sweep_takes_other_parts_than_its_engines(gpu, dim, spec):
    """A sweep chooses parts by the tiles of all its systems, an engine by its
    own: the same fields bit for bit where the windows exceed a list."""
    import torch

    fields = ("virial", "kinetic")
    systems = []
    for q, (N, nf, side) in enumerate(spec):
        frames = _frames(dim, N, nf, 13000 + 100 * q)
        e = engine.Engine(dim=dim, max_rcut=RMAX)
        e.set_gather_mode("tile")
        e.set_box(frames[0]["L"], frames[0]["periodic"])
        e.set_grid(_grid("lattice", frames[0]["L"][0], dim, side))
        y = {"engine": e, "nframes": nf, "n": N, "frames": frames}
        y.update({k: _stack(frames, k) for k in ("pos", "diam", "mass", "vel")})
        y.update({k: torch.full((nf, e.G, dim, dim), np.nan, dtype=torch.float64, device="cuda") for k in fields})
        systems.append(y)
    torch.cuda.synchronize()
    print("sweep of %s" % (spec,), flush=True)
    engine.Sweep(systems, fields=fields).run()
    for q, y in enumerate(systems):
        for f in range(min(3, y["nframes"])):
            one = _fields(y["engine"], y["frames"], fields, first=f, count=1)
            for k in fields:
                assert np.array_equal(y[k][f].cpu().numpy(), one[k][0]), (q, f, k)


@pytest.mark.parametrize("members", [249, 250, 256])
def test_an_enqueued_job_repeats_the_one_that_grew_its_capacity(gpu, members):
    """A cluster whose particles have 248, 249 or 255 bonds, for which the bond
    capacity grows to 248 or 256 slots, on both sides of the tile gather's 255:
    the enqueued job takes the gather that the growing one took, so the same
    bits."""
    import torch

    N = 700
    s = _frames(2, N, 1, 14000)[0]
    # the cluster: a square lattice of spacing 0.05 inside every pair's cutoff
    # (1.25 x 0.73), in place of `members` particles
    q = np.argsort(np.abs(s["pos"]).max(1))[:members]
    s["pos"][q, 0], s["pos"][q, 1] = 0.05 * (np.arange(members) % 16 - 7.5), 0.05 * (np.arange(members) // 16 - 7.5)
    s["pos"][q, :2] *= 0.5
    s["pos"][q, :2] += 1e-3 * np.random.default_rng(1).normal(size=(members, 2))
    far = np.setdiff1d(np.nonzero(np.abs(s["pos"][:, :2]).max(1) < 4.0)[0], q)
    s["pos"][far, :2] += 8.0
    e = engine.Engine(dim=2, max_rcut=RMAX)
    e.set_box(s["L"], s["periodic"])
    e.set_grid(_grid("lattice", s["L"][0], 2, 33))
    grown = _fields(e, [s], ("virial",))["virial"]
    st = e.stats()
    print("enqueue after growth: members %d, most bonds %d, capacity %d" % (members, st["max_bonds"], st["bond_capacity"]),
          flush=True)
    assert members - 1 <= st["max_bonds"] <= 255 and st["bond_capacity"] == (248 if members == 249 else 256)
    out = torch.full((1, e.G, 2, 2), np.nan, dtype=torch.float64, device="cuda")
    pos, diam = _stack([s], "pos"), _stack([s], "diam")
    torch.cuda.synchronize()
    e.enqueue_frames(1, N, pos, diam, fields=("virial",), d_virial=out)
    e.finish()
    assert np.array_equal(out.cpu().numpy(), grown)


def test_more_frames_than_a_launch_takes(gpu):
    """70,000 frames of 20 particles on 16 points, launch settings untouched:
    more frames than a launch's y extent holds (65,535), far fewer particles
    than fill it.  Frames repeat a few, whose fields they must have."""
    import torch

    N, nf, kinds = 20, 70000, 5
    frames = _frames(2, N, kinds, 15000)
    e = engine.Engine(dim=2, max_rcut=RMAX)
    e.set_box(frames[0]["L"], frames[0]["periodic"])
    e.set_grid(_grid("lattice", frames[0]["L"][0], 2, 4))
    few = _fields(e, frames, ("virial", "kinetic"))
    t = {k: _stack(frames, k).repeat(nf // kinds, *([1] * (frames[0][k].ndim))) for k in ("pos", "diam", "mass", "vel")}
    out = {k: torch.full((nf, 16, 2, 2), np.nan, dtype=torch.float64, device="cuda") for k in few}
    torch.cuda.synchronize()
    print("70,000 frames", flush=True)
    e.compute_frames(nf, N, t["pos"], t["diam"], t["mass"], t["vel"], fields=("virial", "kinetic"),
                     **{"d_" + k: v for k, v in out.items()})
    torch.cuda.synchronize()
    for k, v in out.items():
        ref = torch.tensor(few[k], device="cuda").repeat(nf // kinds, 1, 1, 1)
        assert torch.equal(v, ref), k


@pytest.mark.parametrize("kind", ["dense", "wide"])
def test_a_job_keeps_to_its_work_memory(gpu, kind):
    """Launch settings untouched.  dense: 1,500 frames of 400 particles that are
    all bonded to one another (400 slots of 24 bytes each: 5.8 GB of entries in
    one launch).  wide: 3,000 frames of 30 particles in a box of 740 x 740 cells
    (6.6 GB of cell starts).  Both fit the 4 GB of a launch in two or three of
    them, with the fields of frames on their own."""
    import torch

    N, nf, kinds = (400, 1500, 3) if kind == "dense" else (30, 3000, 3)
    frames = _frames(2, N, kinds, 16000)
    L = frames[0]["L"] * (1.0 if kind == "dense" else 1500.0 / frames[0]["L"][0])
    if kind == "dense":
        for s in frames:
            s["pos"][:, :2] = 0.02 * s["pos"][:, :2] + L[:2] / 6  # about a grid point
    e = engine.Engine(dim=2, max_rcut=RMAX)
    e.set_box([L[0], L[1], 1.0], [1, 1, 0])
    e.set_grid(_grid("lattice", frames[0]["L"][0], 2, 4))
    ones = [_fields(e, frames, ("virial",), first=f, count=1)["virial"][0] for f in range(kinds)]
    e.close()
    e = engine.Engine(dim=2, max_rcut=RMAX)
    e.set_box([L[0], L[1], 1.0], [1, 1, 0])
    e.set_grid(_grid("lattice", frames[0]["L"][0], 2, 4))
    pos, diam = (_stack(frames, k).repeat(nf // kinds, *([1] * (frames[0][k].ndim))) for k in ("pos", "diam"))
    out = torch.full((nf, 16, 2, 2), np.nan, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    e.compute_frames(nf, N, pos, diam, fields=("virial",), d_virial=out)
    torch.cuda.synchronize()
    took = (free - torch.cuda.mem_get_info()[0]) / 2 ** 30
    print("%s: capacity %d, work memory %.2f GB" % (kind, e.stats()["bond_capacity"], took), flush=True)
    assert e.stats()["bond_capacity"] >= (400 if kind == "dense" else 16)
    assert took <= 4.2 and out.abs().max() > 0
    assert torch.equal(out, torch.tensor(np.stack(ones), device="cuda").repeat(nf // kinds, 1, 1, 1))


@pytest.mark.parametrize("N,side,nf", [(2000, 24, 5), (4096, 256, 3)])
def test_a_sized_engine_takes_fewer_frames(gpu, N, side, nf):
    """Fewer frames make more wavefronts: quarter blocks of the bond kernel (5
    frames of 2,000 particles 160 blocks, 4 of them 500), smaller parts of the
    tiles (3 frames of 1,024 tiles 3,072 whole ones, one 4,096 quarters).  An
    engine sized by the larger job enqueues the smaller ones, and computes them
    while its buffers are held."""
    import torch

    frames = _frames(2, N, nf, 17000)
    fresh = engine.Engine(dim=2, max_rcut=RMAX)
    e = engine.Engine(dim=2, max_rcut=RMAX)
    for x in (fresh, e):
        x.set_box(frames[0]["L"], frames[0]["periodic"])
        x.set_grid(_grid("lattice", frames[0]["L"][0], 2, side))
    ref = _fields(fresh, frames, ("virial",))["virial"]
    print("fewer frames: N=%d side %d, %d frames" % (N, side, nf), flush=True)
    assert np.array_equal(_fields(e, frames, ("virial",))["virial"], ref)
    pos, diam = _stack(frames, "pos"), _stack(frames, "diam")
    for m in range(nf, 0, -1):
        out = torch.full((m, e.G, 2, 2), np.nan, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        e.enqueue_frames(m, N, pos[:m], diam[:m], fields=("virial",), d_virial=out)
        e.finish()
        assert np.array_equal(out.cpu().numpy(), ref[:m]), m
        assert np.array_equal(_fields(e, frames, ("virial",), count=m)["virial"], ref[:m]), m
    e.set_gather_mode("lane")  # and after a change of gather
    assert np.isfinite(_fields(e, frames, ("virial",))["virial"]).all()
    e.release_enqueued()


def test_a_sized_engine_takes_more_frames(gpu):
    """An engine sized by eight frames, launch settings untouched, enqueues 37
    of them and computes 37 while its buffers are held: in launches that the
    buffers hold, the same fields.  Sized by five, it refuses eight."""
    import torch

    N, nf = 1500, 37
    frames = _frames(2, N, nf, 18000)
    fresh = engine.Engine(dim=2, max_rcut=RMAX)
    e = engine.Engine(dim=2, max_rcut=RMAX)
    for x in (fresh, e):
        x.set_box(frames[0]["L"], frames[0]["periodic"])
        x.set_grid(_grid("lattice", frames[0]["L"][0], 2, 24))
    ref = _fields(fresh, frames, ("virial", "kinetic"))
    pos, diam, mass, vel = (_stack(frames, k) for k in ("pos", "diam", "mass", "vel"))

    def enqueue(m):
        out = {k: torch.full((m, e.G, 2, 2), np.nan, dtype=torch.float64, device="cuda") for k in ref}
        torch.cuda.synchronize()
        e.enqueue_frames(m, N, pos[:m], diam[:m], mass[:m], vel[:m], fields=("virial", "kinetic"),
                         **{"d_" + k: v for k, v in out.items()})
        e.finish()
        return {k: v.cpu().numpy() for k, v in out.items()}

    _fields(e, frames, ("virial", "kinetic"), count=5)
    with pytest.raises(engine.PGTError, match="PGT_ERR_STATE"):
        enqueue(8)
    _fields(e, frames, ("virial", "kinetic"), count=8)
    print("more frames: 8, then 37", flush=True)
    for got in (enqueue(nf), _fields(e, frames, ("virial", "kinetic")), enqueue(8)):
        for k in ref:
            assert np.array_equal(got[k], ref[k][:len(got[k])]), k
    e.release_enqueued()


def test_noalloc_of_a_dense_system_runs_once(gpu):
    """Particles with more than 255 bonds: once the no-allocation entry point
    has found their capacity, an engine whose gather was not chosen goes to the
    lane gather at once, as one told to (the shortest of 15 calls within 1.25
    times the other's; a job that runs with the tile gather first takes 1.5
    times as long)."""
    import time
    import torch

    import oracle

    N, rc = 2500, 10.0
    s = workload.make_system(N, 2, 19000)
    pos, diam = _stack([s], "pos"), _stack([s], "diam")
    took, got = {}, {}
    for mode in ("lane", None):
        e = engine.Engine(dim=2, params=oracle.poly12_params(rcut=rc), scaled_rcut=rc, max_rcut=rc * float(s["diam"].max()))
        if mode:
            e.set_gather_mode(mode)
        e.set_box(s["L"], s["periodic"])
        e.set_grid(_grid("lattice", s["L"][0], 2, 48))
        out = torch.full((1, e.G, 2, 2), np.nan, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        times = []
        for _ in range(18):
            t = time.perf_counter()
            e.compute_frames_noalloc(1, N, pos, diam, fields=("virial",), d_virial=out)
            times.append(time.perf_counter() - t)
        assert e.stats()["max_bonds"] > 255
        took[mode], got[mode] = min(times[3:]), out.cpu().numpy()
    print("noalloc, dense: lane %.2f ms, by default %.2f ms" % (1e3 * took["lane"], 1e3 * took[None]), flush=True)
    assert np.array_equal(got[None], got["lane"])
    assert took[None] <= 1.25 * took["lane"]


@pytest.mark.parametrize("dim,N,nf,periodic,squeeze", [
    (2, 41, 1, (0, 0, 0), 1.0), (2, 1000, 1, (0, 0, 0), 1.0), (2, 8192, 2, (0, 0, 0), 1.0), (2, 8191, 1, (1, 0, 0), 1.0),
    (2, 8192, 1, (1, 1, 0), 0.25), (2, 3001, 3, (1, 1, 0), 0.02), (3, 8192, 1, (0, 0, 0), 1.0), (3, 8100, 1, (1, 0, 0), 1.0),
    (3, 8192, 1, (1, 1, 1), 0.1), (3, 1025, 2, (1, 1, 1), 0.3)])
def test_crowded_small_frames_keep_their_order(gpu, dim, N, nf, periodic, squeeze):
    """Frames of up to 8,192 particles with crowded cells: boxes of one cell,
    of a row of cells, of a plane of them, clusters in a periodic box of more
    than 128 cells.  The lane gather adds the kinetic terms in the order of the
    cell list: bit for bit those of the same frames with particles far from the
    grid added until they are sorted by the launches of larger frames.  And in
    good time (a box of one cell once took 3 ms)."""
    import time
    import torch

    frames = _frames(dim, N, nf, 20000)
    L = np.array([90.0, 90.0, 1.0]) if dim == 2 else np.array([30.0, 30.0, 30.0])
    rng = np.random.default_rng(5)
    more = 8193 - N + 100
    larger = []
    for s in frames:
        s["pos"][:, :dim] *= squeeze * 0.4 * L[0] / s["L"][0]
        far = {"pos": np.zeros((more, 3)), "diam": np.ones(more), "mass": np.ones(more), "vel": rng.normal(size=(more, 3))}
        far["pos"][:, :dim] = rng.uniform(0.38, 0.42, (more, dim)) * L[:dim]
        larger.append({k: np.concatenate([s[k], far[k]]) for k in far})
    grid = _grid("lattice", 0.3 * L[0] * squeeze, dim, 9 if dim == 2 else 5)
    print("crowded %dD N=%d x %d %s squeeze %.2f" % (dim, N, nf, periodic, squeeze), flush=True)
    got = []
    for x in (frames, larger):
        e = engine.Engine(dim=dim, max_rcut=RMAX)
        e.set_gather_mode("lane")
        e.set_box(L, periodic)
        e.set_grid(grid)
        got.append((_fields(e, x, ("kinetic",))["kinetic"], e.stats()["n_ball"]))
        if x is frames:
            out = torch.empty((nf, e.G, dim, dim), dtype=torch.float64, device="cuda")
            args = [_stack(x, k) for k in ("pos", "diam", "mass", "vel")]
            torch.cuda.synchronize()
            times = []
            for _ in range(10):
                t = time.perf_counter()
                e.compute_frames(nf, N, *args, fields=("kinetic",), d_kinetic=out)
                times.append(time.perf_counter() - t - 1e-3 * e.stats()["gather_ms"])
    assert got[0][1] == got[1][1] > 0
    assert np.isfinite(got[0][0]).all() and np.array_equal(got[0][0], got[1][0])
    print("  without the gather %.0f us" % (1e6 * min(times)), flush=True)
    assert min(times) < 8e-4


def test_a_closed_engine_gives_its_interval_tables_back(gpu):
    """An adaptive job whose integrals outgrow the private tables takes tables
    of the caller's limit (0.9 GB here) from device memory, which closing the
    engine gives back."""
    import torch

    s, grid = workload.config_frame(1, 2)
    torch.cuda.synchronize()
    for k in range(2):  # (the first engine loads code and tables of the runtime's)
        before = torch.cuda.mem_get_info()[0]
        e = engine.Engine(dim=2, cg="rect", max_rcut=RMAX, adaptive=(900, 0.0, 0.0))
        e.set_system(s, grid)
        e.compute(fields=("virial",))
        took = before - torch.cuda.mem_get_info()[0]
        e.close()
        left = before - torch.cuda.mem_get_info()[0]
        print("interval tables: took %.2f GB, kept %.3f GB" % (took / 2 ** 30, left / 2 ** 30), flush=True)
    assert took > 5e8
    assert left < 1e8


@pytest.mark.parametrize("kind", ["scattered", "row"])
def test_tiles_off_a_lattice_keep_to_their_surroundings(gpu, kind):
    """Points off a lattice leave lanes of a tile without a point: the tile's
    window is that of its points.  On 40,000 particles a window that reaches to
    the middle of the box took 0.62 and 0.22 ms, one about the points 0.05 and 0.01."""
    N = 40000
    s = workload.make_system(N, 2, 21000)
    L = s["L"][0]
    grid = (np.random.default_rng(8).uniform(-0.5 * L, 0.5 * L, (3000, 3)) * [1, 1, 0] if kind == "scattered"
            else np.linspace(-0.5, 0.5, 3000)[:, None] * [L, 0.3 * L, 0])
    e = engine.Engine(dim=2, max_rcut=RMAX)
    e.set_system(s, grid)
    took = []
    for _ in range(8):
        e.compute(("virial",))
        took.append(e.stats()["gather_ms"])
    print("off a lattice, %s: gather %.3f ms" % (kind, min(took)), flush=True)
    assert min(took) < 0.15
