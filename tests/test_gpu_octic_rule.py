"""Rounding of the tile gather's 5-node Octic rule against long double."""
import numpy as np
import pytest

from pyglasstools_amd import engine

pytestmark = pytest.mark.gpu


def _rule():
    """Nodes and weights of the rule on [0, 1] in long double."""
    x = np.polynomial.legendre.leggauss(5)[0].astype(np.longdouble)
    for _ in range(4):
        x = x - (63 * x ** 5 - 70 * x ** 3 + 15 * x) / (315 * x ** 4 - 210 * x ** 2 + 15)
    d = (315 * x ** 4 - 210 * x ** 2 + 15) / 8
    return (x + 1) / 2, 1 / ((1 - x * x) * d * d)


def test_tile_rule_rounds_no_more_than_the_lane_gathers(gpu):
    """One bond seen from 20,000 points whose balls hold one of its ends.
    Coordinates are multiples of 2^-9 and the radius is 2, so that everything
    before the rule is exact; the force is the same factor for every point, and
    there is nothing to add.  What is left are the roundings of the rule and of
    the products after it, which the gathers share: the root mean square of the
    tile gather's error may not exceed the lane gather's by more than its
    uncertainty (1/sqrt(2 x 20,000) of either, twice that and some: 2%)."""
    u = 2.0 ** -9
    rng = np.random.default_rng(2)
    pos = np.array([[3 * u, -7 * u, 0.0], [3 * u + 401 * u, -7 * u + 308 * u, 0.0]])
    diam = np.array([1.0, 1.0])
    pts = np.zeros((120000, 3))
    pts[:, :2] = pos[0, :2] + u * rng.integers(-1024, 1024, (120000, 2))
    r2 = [((pts - p)[:, :2] ** 2).sum(1) for p in pos]
    pts = pts[(r2[0] < 3.99) & (r2[1] > 4.01)][:20000]
    b = (pos[1] - pos[0])[:2].astype(np.longdouble)
    s, w = _rule()
    ref = 0
    a = (pos[0, :2] - pts[:, :2]).astype(np.longdouble)
    for sk, wk in zip(s, w):
        t = ((a + sk * b) ** 2).sum(1) / 4
        ref = ref + wk * np.maximum(1 - t * t, 0) ** 2
    rms = {}
    for mode in ("lane", "tile"):
        e = engine.Engine(dim=2, max_rcut=1.25)
        e.set_gather_mode(mode)
        e.set_box([64.0, 64.0, 1.0], [1, 1, 0])
        e.set_particles(pos, diam)
        e.set_grid(pts)
        T = e.compute(fields=("virial",))["virial"].astype(np.longdouble)
        err = []
        for i, j in ((0, 0), (1, 1), (0, 1)):
            K = (T[:, i, j] * ref).sum() / (ref * ref).sum()  # the force's factor
            err.append(T[:, i, j] / K - ref)
        rms[mode] = float(np.sqrt(np.mean(np.square(err))))
    print("rms error of the rule, %d points: lane %.3e, tile %.3e" % (len(pts), rms["lane"], rms["tile"]), flush=True)
    assert len(pts) == 20000 and 1e-17 < rms["lane"] < 4e-16
    assert rms["tile"] <= 1.02 * rms["lane"]
