"""The form for fp64 sums too small to fill the chip (below 4,096 pairs of 512 targets and a
256-source tile on 256 compute units), at the ends of its chunks (64 sources), target sets (256)
and at the line where it begins, against the oracle.

The bar is the fp64 form's own, 1e-12 relative L2. The oracle's
vorticity factor 2 K + bbb d^2 cancels far from a core (one pair of the WL core at d^2 = 593 w: 3e-11
off in 64 bits), so the algebraic cores' sums are taken in 80 bits, that factor in closed form."""
import numpy as np
import pytest
import torch

import oracle as O
import omega2d_amd as o2d
from helpers import particles, rel_l2

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (3, 255), (63, 256), (64, 257), (65, 1), (255, 700), (256, 63), (257, 64),
         (4097, 65), (70000, 5), (9, 30001)]


def sums(core, sx, sy, ss, sr, tx, ty, tr, results):
    if core == "gauss":
        return O.points_on_points(core, sx, sy, ss, sr, tx, ty, tr, results)
    sx, sy, ss, sr, tx, ty = (np.asarray(a, np.longdouble) for a in (sx, sy, ss, sr, tx, ty))
    tr = np.zeros(len(tx), np.longdouble) if tr is None else np.asarray(tr, np.longdouble)
    power = {"rm": 2, "wl": 2, "v2": 4, "v3": 6}[core]
    dx, dy = tx[:, None] - sx, ty[:, None] - sy
    d2, w = dx * dx + dy * dy, sr**power + tr[:, None]**power
    if core == "rm":
        k = 1 / (d2 + w)
        b, vort = -2 * k * k, 2 * w * k * k
    elif core == "wl":
        k = (d2 + 2 * w) / (d2 + w)**2
        b, vort = (2 - 4 * k * (d2 + w)) / (d2 + w)**2, 4 * w * w / (d2 + w)**3
    elif core == "v2":
        k = 1 / np.sqrt(d2 * d2 + w)
        b, vort = -2 * k**3 * d2, 2 * w * k**3
    else:
        k = 1 / np.cbrt(d2**3 + w)
        b, vort = -2 * d2 * d2 * k**4, 2 * w * k**4
    out = [-(ss * k * dy).sum(1), (ss * k * dx).sum(1)]
    if results == "vort":
        out.append((ss * vort).sum(1))
    elif results == "shear":
        out.append((abs(ss * b) * d2).sum(1) / 2)
    return [o.astype(float) for o in out]


@pytest.mark.parametrize("precision,bar", [("fp64", 1e-12)])
@pytest.mark.parametrize("core", ["rm", "gauss", "wl", "v2", "v3"])
@pytest.mark.parametrize("ns,nt", SIZES)
def test_small_sums_match_oracle(ns, nt, core, precision, bar):
    rng = np.random.default_rng(ns + nt)
    sx, sy, ss, sr = particles(rng, ns, rad=(0.01, 0.3))
    tx, ty, _, tr = particles(rng, nt, rad=(0.01, 0.3))
    for results, radius in (("vel", None), ("vort", tr), ("shear", np.full(nt, 0.1))):
        got = o2d.points_on_points(sx, sy, ss, sr, tx, ty, radius, core=core, results=results,
                                   precision=precision)
        ref = sums(core, sx, sy, ss, sr, tx, ty, radius, results)
        for g, r in zip(got, ref):
            assert rel_l2(g, r) <= bar, (results, rel_l2(g, r))


@pytest.mark.parametrize("precision,bar,size", [("fp64", 1e-12, 512)])
@pytest.mark.parametrize("core", ["rm", "gauss"])
def test_both_sides_of_the_line(core, precision, bar, size):
    """One source more or less than the line: the two forms agree with the oracle on the last 200
    targets and with each other (the source that only one of them has is of zero strength)."""
    tiles = 16 * torch.cuda.get_device_properties(0).multi_processor_count
    nt = 64 * size
    ns = 256 * ((tiles + 63) // 64 - 1)  # the most that is still small
    rng = np.random.default_rng(5)
    sx, sy, ss, sr = particles(rng, ns + 1, rad=(0.005, 0.05))
    ss[-1] = 0.0
    tx, ty, _, tr = particles(rng, nt, rad=(0.005, 0.05))
    small = o2d.points_on_points(sx[:-1], sy[:-1], ss[:-1], sr[:-1], tx, ty, tr, core=core,
                                 precision=precision)
    large = o2d.points_on_points(sx, sy, ss, sr, tx, ty, tr, core=core, precision=precision)
    ref = O.points_on_points(core, sx, sy, ss, sr, tx[-200:], ty[-200:], tr[-200:])
    for a, b, r in zip(small, large, ref):
        assert rel_l2(a, b) <= 2 * bar
        assert rel_l2(a[-200:], r) <= bar and rel_l2(b[-200:], r) <= bar
