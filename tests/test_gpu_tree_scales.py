"""Cluster sums at coordinate scales where the squares of a cell's radius and distance leave the range
of a float (and on both sides of it): the orders a far cell needs depend on their quotient only, so a
scaled problem has the scaled answer. 1e-12 relative L2 where the series are exact to rounding, the
fp64 form's bar; the treecode at (0.4, 30) within its 1e-10."""
import numpy as np
import pytest
import torch

import oracle as O
from helpers import rel_l2
from omega2d_amd import device as dv

pytestmark = pytest.mark.gpu

SCALES = [1e-60, 1e-23, 1e-22, 1e-21, 1e-19, 1e-10, 1e10, 1e18, 1e19, 1e20, 1e21, 1e60]


def T(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def blobs(rng, n):
    c, b = rng.uniform(-2, 2, (7, 2)), rng.integers(0, 7, n)
    return c[b, 0] + 0.05 * rng.normal(size=n), c[b, 1] + 0.05 * rng.normal(size=n)


@pytest.mark.parametrize("scale", SCALES)
def test_velocity_and_treecode_scale(scale):
    rng = np.random.default_rng(3)
    n = 20000  # 4e8 pairs: far sources by clusters
    x, y = blobs(rng, n)
    s, r = rng.normal(size=n), np.full(n, 1e-3)
    at = np.arange(0, n, 50)
    exact = np.concatenate(O.points_on_points("gauss", x, y, s, r, x[at], y[at], r[at]))
    d = [T(x * scale), T(y * scale), T(s), T(r * scale)]
    sub = torch.from_numpy(at).cuda()
    for got, bar in ((dv.points_on_points(*d, d[0], d[1], d[3], core="gauss", precision="fp64"), 1e-12),
                     (dv.points_on_points_tree(*d, d[0], d[1], d[3], core="gauss", theta=0.4,
                                               order=30), 1e-10)):
        assert rel_l2(torch.cat([g[sub] for g in got]).cpu().numpy() * scale, exact) <= bar


@pytest.mark.parametrize("scale", SCALES)
def test_adjoint_scales(scale):
    rng = np.random.default_rng(4)
    ns, nt = 50001, 4096
    x, y = blobs(rng, ns)
    s, r = rng.normal(size=ns), np.full(ns, 1e-3)
    tx, ty = blobs(rng, nt)
    gu, gv = rng.normal(size=nt), rng.normal(size=nt)
    got = dv.points_on_points_adjoint(T(x * scale), T(y * scale), T(s), T(r * scale), T(tx * scale),
                                      T(ty * scale), T(gu), T(gv), core="gauss")
    at = np.arange(0, ns, 150)
    ref = O.points_on_points_adjoint("gauss", x[at], y[at], s[at], r[at], tx, ty, gu, gv)
    for g, e, power in zip(got, ref, (2, 2, 1, 2)):  # d/dx, d/dy and d/dr shrink twice as fast
        assert rel_l2(g.cpu().numpy()[at] * scale**power, e) <= 1e-12
