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
