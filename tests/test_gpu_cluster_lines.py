"""The lines between the pair by pair and the clustered fp64 Gaussian sums: shapes on both sides of them
(few targets among many sources, few sources, the adjoint of few particles or probes), and calls whose
cores hold so much of the set that the device turns them back to pairs, against the oracle at the fp64
form's 1e-12 relative L2."""
import numpy as np
import pytest
import torch

import oracle as O
from helpers import rel_l2
from omega2d_amd import device as dv

pytestmark = pytest.mark.gpu


def T(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def blobs(rng, n):
    c, b = rng.uniform(-2, 2, (7, 2)), rng.integers(0, 7, n)
    return c[b, 0] + 0.1 * rng.normal(size=n), c[b, 1] + 0.1 * rng.normal(size=n)


def radii(rng, n, wide):
    r = rng.uniform(0.001, 0.01, n)
    if wide == "all":
        r += 2.0
    elif wide == "some":  # cores that reach a tenth of the set or all of it
        r[rng.uniform(size=n) < 0.3] = 0.5
    elif wide == "one":
        r[n // 2] = 3.0
    return r


def few(n):
    return np.unique(np.linspace(0, n - 1, 100).astype(np.int64))


@pytest.mark.parametrize("wide", ["none", "one", "some", "all"])
@pytest.mark.parametrize("ns,nt", [(20011, 20011), (700001, 40), (1500001, 40), (300001, 1000),
                                   (300001, 2049), (40001, 9001), (999, 400001), (33, 3000001)])
def test_velocity(ns, nt, wide):
    rng = np.random.default_rng(ns + nt)
    x, y = blobs(rng, ns)
    s, r = rng.normal(size=ns), radii(rng, ns, wide)
    d = [T(a) for a in (x, y, s, r)]
    if ns == nt:
        tx, ty, tr, dt, dr = x, y, r, d[:2], d[3]
    else:
        tx, ty = blobs(rng, nt)
        tr = radii(rng, nt, wide) if nt % 4 == 1 else None
        dt, dr = [T(tx), T(ty)], None if tr is None else T(tr)
    at = few(nt)
    u0, v0 = rng.normal(size=nt), rng.normal(size=nt)
    got = dv.points_on_points(*d, *dt, dr, core="gauss", precision="fp64", tu=T(u0), tv=T(v0))
    ref = O.points_on_points("gauss", x, y, s, r, tx[at], ty[at], None if tr is None else tr[at])
    a = np.concatenate([g.cpu().numpy()[at] for g in got])
    assert rel_l2(a, np.concatenate([u0[at] + ref[0], v0[at] + ref[1]])) <= 1e-12


@pytest.mark.parametrize("wide", ["none", "one", "some", "all"])
@pytest.mark.parametrize("ns,nt", [(20011, 20011), (100003, 2500), (100003, 3001), (1000001, 300),
                                   (1000001, 700), (9001, 60001), (3001, 150001), (1001, 1000001),
                                   (33, 700001)])
def test_adjoint(ns, nt, wide):
    rng = np.random.default_rng(ns + nt)
    x, y = blobs(rng, ns)
    s, r = rng.normal(size=ns), radii(rng, ns, wide)
    tx, ty = blobs(rng, nt)
    gu, gv = rng.normal(size=nt), rng.normal(size=nt)
    got = dv.points_on_points_adjoint(*[T(a) for a in (x, y, s, r, tx, ty, gu, gv)], core="gauss")
    at = few(ns)
    ref = O.points_on_points_adjoint("gauss", x[at], y[at], s[at], r[at], tx, ty, gu, gv)
    for g, e in zip(got, ref):
        assert rel_l2(g.cpu().numpy()[at], e) <= 1e-12
