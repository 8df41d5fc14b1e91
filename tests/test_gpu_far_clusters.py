"""The fp64 Gaussian velocity sum and its adjoint from 3.5e8 and 2e8 pairs, where far sources are
taken by clusters, against the oracle and against the pair by pair sum of the no-allocation entry.

The bar is the fp64 form's, 1e-12 relative L2 (a far cluster's remainder is below 6e-16 of its
sum of magnitudes). Sizes sit at the edges of the groups: 64 or 16 targets per wave (16 from four
times as many sources as targets), 1,024 targets per super group (used from 16 of them), 32
sources per leaf, four cells per parent."""
import ctypes

import numpy as np
import pytest
import torch

import oracle as O
from helpers import rel_l2
from omega2d_amd import _cabi
from omega2d_amd import device as dv
from omega2d_amd.device import env_for

pytestmark = pytest.mark.gpu

BAR = 1e-12


def T(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def layout(rng, n, kind):
    """Positions: blobs with a few far outliers (the Morton curve jumps between them), a uniform
    square, or one line of coincident pairs."""
    if kind == "blobs":
        c = rng.uniform(-2, 2, (7, 2))
        b = rng.integers(0, 7, n)
        x, y = c[b, 0] + 0.05 * rng.normal(size=n), c[b, 1] + 0.05 * rng.normal(size=n)
        x[:5] = 40.0 * rng.normal(size=5)
    elif kind == "square":
        x, y = rng.uniform(-1, 1, n), rng.uniform(-1, 1, n)
    else:
        x, y = np.repeat(rng.uniform(-1, 1, (n + 1) // 2), 2)[:n], np.zeros(n)
    return x, y


def pair_by_pair(src, tgt, tr):
    """The direct sum (o2d_hip_points_on_points_noalloc_dev_d never takes clusters)."""
    s, t = [T(a) for a in src], [T(a) for a in tgt]
    u = torch.zeros(len(tgt[0]), dtype=torch.float64, device="cuda")
    v = torch.zeros_like(u)
    env = env_for(u.device, "gauss", "fp64", "vel")
    r = None if tr is None else T(tr)
    p = lambda a: None if a is None else ctypes.c_void_p(a.data_ptr())  # noqa: E731
    _cabi.call("o2d_hip_points_on_points_noalloc_dev_d", ctypes.byref(env), len(src[0]),
               *[p(a) for a in s], len(tgt[0]), *[p(a) for a in t], p(r), p(u), p(v), None, None)
    torch.cuda.synchronize()
    return u.cpu().numpy(), v.cpu().numpy()


def clusters(src, tgt, tr, tu=None, tv=None):
    s = [T(a) for a in src]
    t = s[:2] if tgt is None else [T(a) for a in tgt]
    r = s[3] if isinstance(tr, str) else (None if tr is None else T(tr))
    u, v = dv.points_on_points(*s, *t, r, core="gauss", precision="fp64",
                               tu=None if tu is None else T(tu), tv=None if tv is None else T(tv))
    torch.cuda.synchronize()
    return u.cpu().numpy(), v.cpu().numpy()


@pytest.mark.parametrize("kind", ["blobs", "square", "line"])
@pytest.mark.parametrize("sigma", [1e-4, (0.002, 0.03)])
@pytest.mark.parametrize("ns,nt", [(18719, None), (22033, 16384), (21377, 16385), (65537, 16383),
                                   (131075, 3111), (262144, 1601), (1601, 262144)])
def test_clusters_match_pairs(ns, nt, sigma, kind):
    rng = np.random.default_rng(ns)
    draw = lambda n: (np.full(n, sigma) if np.isscalar(sigma)  # noqa: E731
                      else rng.uniform(*sigma, n))
    x, y = layout(rng, ns, kind)
    src = (x, y, rng.normal(0, 1e-3, ns), draw(ns))
    if nt is None:  # on themselves: sources and targets share one order and one set of records
        got, tgt, tr = clusters(src, None, "self"), src[:2], src[3]
    else:
        tgt = layout(rng, nt, "square" if kind == "line" else kind)
        tr = draw(nt) if nt % 2 else None
        got = clusters(src, tgt, tr)
    ref = pair_by_pair(src, tgt, tr)
    assert rel_l2(np.concatenate(got), np.concatenate(ref)) <= BAR
    sub = np.arange(0, len(tgt[0]), max(1, len(tgt[0]) // 200))
    exact = O.points_on_points("gauss", *src, tgt[0][sub], tgt[1][sub],
                               None if tr is None else tr[sub])
    assert rel_l2(np.concatenate([g[sub] for g in got]), np.concatenate(exact)) <= BAR


@pytest.mark.parametrize("scale", [1e-60, 1e60])
def test_scaled_problem_scales(scale):
    # cluster moments are taken relative to the cluster's radius: no power over- or underflows
    rng = np.random.default_rng(3)
    x, y = layout(rng, 20000, "blobs")
    s, r = rng.normal(size=20000), np.full(20000, 1e-3)
    a = clusters((x, y, s, r), None, "self")
    b = clusters((x * scale, y * scale, s, r * scale), None, "self")
    assert rel_l2(np.concatenate(b) * scale, np.concatenate(a)) <= BAR


def test_accumulates_and_all_points_coincide():
    rng = np.random.default_rng(4)
    n = 19000
    src = (np.full(n, 0.5), np.full(n, -0.25), rng.normal(size=n), np.full(n, 0.01))
    t0 = rng.normal(size=n), rng.normal(size=n)
    u, v = clusters(src, (rng.uniform(1, 2, n), rng.uniform(1, 2, n)), None, *t0)
    assert np.all(np.isfinite(u)) and not np.array_equal(u, t0[0])
    u, v = clusters(src, None, "self", *t0)  # every pair at distance 0 adds exactly 0
    assert np.array_equal(u, t0[0]) and np.array_equal(v, t0[1])


@pytest.mark.parametrize("what", ["strength", "source", "target", "source radius",
                                  "target radius"])
@pytest.mark.parametrize("value", [np.inf, np.nan])
def test_values_that_are_not_finite(what, value):
    """One of them reaches the same sums as pair by pair, and no others. (A NaN source radius makes
    NaN where a tile or leaf is near enough to be tested pair by pair, which is not the same set
    in both; elsewhere neither sum looks at it.)"""
    rng = np.random.default_rng(6)
    ns, nt = 19100, 19200
    src = [*layout(rng, ns, "blobs"), rng.normal(size=ns), np.full(ns, 1e-3)]
    tgt, tr = list(layout(rng, nt, "blobs")), np.full(nt, 1e-3)
    {"strength": src[2], "source": src[0], "target": tgt[1], "source radius": src[3],
     "target radius": tr}[what][777] = value
    got, ref = clusters(src, tgt, tr), pair_by_pair(src, tgt, tr)
    for g, r in zip(got, ref):
        if what == "source radius" and np.isnan(value):
            both = np.isfinite(g) & np.isfinite(r)
            assert both.mean() > 0.5
            assert rel_l2(g[both], r[both]) <= BAR
            continue
        assert np.array_equal(np.isnan(g), np.isnan(r))
        assert np.array_equal(g[np.isinf(r)], r[np.isinf(r)])
        ok = np.isfinite(r)
        if ok.any():
            assert rel_l2(g[ok], r[ok]) <= BAR


@pytest.mark.parametrize("kind", ["blobs", "square"])
@pytest.mark.parametrize("ns,nt", [(50001, 4096), (250000, 801), (3001, 70000)])
def test_adjoint_by_clusters_matches_the_oracle(ns, nt, kind):
    rng = np.random.default_rng(ns + nt)
    x, y = layout(rng, ns, kind)
    s, r = rng.normal(0, 1e-3, ns), rng.uniform(0.002, 0.03, ns)
    tx, ty = layout(rng, nt, kind)
    gu, gv = rng.normal(size=nt), rng.normal(size=nt)
    out = [rng.normal(size=ns) for _ in range(4)]
    got = dv.points_on_points_adjoint(T(x), T(y), T(s), T(r), T(tx), T(ty), T(gu), T(gv),
                                      core="gauss", out=tuple(T(o) for o in out))
    torch.cuda.synchronize()
    sub = np.arange(0, ns, max(1, ns // 300))
    ref = O.points_on_points_adjoint("gauss", x[sub], y[sub], s[sub], r[sub], tx, ty, gu, gv)
    for g, o, e in zip(got, out, ref):
        assert rel_l2(g.cpu().numpy()[sub] - o[sub], e) <= 1e-11  # the outputs' own size comes off
