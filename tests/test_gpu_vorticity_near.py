"""The vorticity sum by boxes of near sources, at the edges of its boxes (32 sources, tiles of 256,
256 listed tiles at a time), its target groups (16, two a workgroup) and its rows of tiles, against
the oracle: 1e-12 relative L2, the sum's own bar."""
import numpy as np
import pytest
import torch

import oracle as O
from helpers import rel_l2
from omega2d_amd import device as dv

pytestmark = pytest.mark.gpu


def T(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def points(rng, n, kind):
    if kind == "sheets":  # thin, dense and far apart
        t = rng.uniform(0, 6, n)
        return t, 0.7 * rng.integers(0, 4, n) + rng.normal(0, 0.01, n)
    return rng.uniform(-1, 1, n), rng.uniform(-1, 1, n)


@pytest.mark.parametrize("kind", ["sheets", "square"])
@pytest.mark.parametrize("ns,nt", [(1, 31), (31, 17), (33, 33), (255, 1), (257, 16), (4096, 1024), (4097, 1025),
                                   (4127, 1039), (4129, 1041), (8225, 1056), (70001, 1057),
                                   (210001, 1100), (5000, 30001)])
def test_near_boxes_match_oracle(ns, nt, kind):
    rng = np.random.default_rng(ns + nt)
    sx, sy = points(rng, ns, kind)
    tx, ty = points(rng, nt, kind)
    ss, sr = rng.normal(size=ns), rng.uniform(0.002, 0.02, ns)
    tw = rng.normal(size=nt)
    got = dv.points_vorticity(T(sx), T(sy), T(ss), T(sr), T(tx), T(ty), tw=T(tw)).cpu().numpy()
    assert rel_l2(got, tw + O.points_vorticity(sx, sy, ss, sr, tx, ty)) <= 1e-12


@pytest.mark.parametrize("n", [4097, 20000])
def test_the_sources_as_targets(n):
    """Targets that are the sources' own arrays share their order: the same sums, bit for bit, as
    with copies of them."""
    rng = np.random.default_rng(n)
    x, y = points(rng, n, "sheets")
    x, y, s, r = T(x), T(y), T(rng.normal(size=n)), T(rng.uniform(0.002, 0.02, n))
    a = dv.points_vorticity(x, y, s, r, x, y)
    b = dv.points_vorticity(x, y, s, r, x.clone(), y.clone())
    assert torch.equal(a, b)
