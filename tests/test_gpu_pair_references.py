"""Full-size sums against references that share no kernel with them: the treecode and the clustered fp64
Gaussian against pair by pair sums on the device, the clustered adjoint against those and the CPU oracle,
and the two fp64 forms on both sides of the line between them, by the entry that never takes clusters."""
import numpy as np
import pytest
import torch

import oracle as O
from helpers import pair_sum, particles, rel_l2
from omega2d_amd import device as dv
from omega2d_amd import workloads as W

pytestmark = pytest.mark.gpu


def T(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def N(pair):
    return np.concatenate([a.cpu().numpy() for a in pair])


def test_tree_and_clusters_on_the_1m_blob_workload():
    w = W.c2_blobs()
    src = [T(w[k]) for k in ("x", "y", "s", "r")]
    trc = [T(w["tx"]), T(w["ty"])]
    m = 4096
    at = torch.arange(0, src[0].numel(), src[0].numel() // m, device="cuda")[:m]
    sub = [a[at].contiguous() for a in (src[0], src[1], src[3])]
    ref = N(pair_sum(src, sub[:2], sub[2]))
    tref = N(pair_sum(src, trc))
    # a sample of the pair by pair reference itself against the CPU oracle
    o = O.points_on_points("gauss", w["x"], w["y"], w["s"], w["r"], w["tx"][:64], w["ty"][:64])
    assert rel_l2(np.concatenate([tref[:64], tref[len(w["tx"]):][:64]]), np.concatenate(o)) <= 1e-12
    for kw, bar in ((dict(theta=0.5, order=20), 1e-7), (dict(theta=0.6, order=28), 1e-9)):
        u, v = dv.points_on_points_tree(*src, src[0], src[1], src[3], core="gauss", **kw)
        assert rel_l2(N((u[at], v[at])), ref) <= bar
        assert rel_l2(N(dv.points_on_points_tree(*src, *trc, None, core="gauss", **kw)), tref) <= bar
    u, v = dv.points_on_points(*src, src[0], src[1], src[3], core="gauss", precision="fp64")
    assert rel_l2(N((u[at], v[at])), ref) <= 1e-12
    assert rel_l2(N(dv.points_on_points(*src, *trc, None, core="gauss", precision="fp64")), tref) <= 1e-12


def test_c4_adjoint_against_the_transposed_pair_sum_and_the_oracle():
    w = W.c4_adjoint()
    d = {k: T(w[k]) for k in ("x", "y", "s", "r", "tx", "ty")}
    src, tgt = [d[k] for k in ("x", "y", "s", "r")], [d["tx"], d["ty"]]
    u, v = pair_sum(src, tgt)
    got = dv.points_on_points(*src, *tgt, None, core="gauss", precision="fp64")
    assert rel_l2(N(got), N((u, v))) <= 1e-12
    rng = np.random.default_rng(5)
    gu, gv = rng.normal(size=len(w["tx"])), rng.normal(size=len(w["tx"]))
    grads = [g.cpu().numpy() for g in dv.points_on_points_adjoint(*src, *tgt, T(gu), T(gv), core="gauss")]
    lhs = float(np.dot(grads[2], w["s"]))
    rhs = float(np.dot(gu, u.cpu().numpy()) + np.dot(gv, v.cpu().numpy()))
    assert abs(lhs - rhs) <= 1e-12 * float(np.dot(np.abs(grads[2]), np.abs(w["s"])))
    at = np.linspace(0, len(w["x"]) - 1, 300).astype(np.int64)
    ref = O.points_on_points_adjoint("gauss", w["x"][at], w["y"][at], w["s"][at], w["r"][at], w["tx"],
                                     w["ty"], gu, gv)
    for g, e in zip(grads, ref):
        assert rel_l2(g[at], e) <= 1e-12


@pytest.mark.parametrize("more", [0, 1])
@pytest.mark.parametrize("core", ["rm", "gauss"])
def test_both_sides_of_the_small_form_pair_by_pair(core, more):
    """The most sources that still make a small sum of 32,768 targets, and one more."""
    tiles = 16 * torch.cuda.get_device_properties(0).multi_processor_count
    nt = 64 * 512
    ns = 256 * ((tiles + 63) // 64 - 1) + more
    rng = np.random.default_rng(5)
    src = particles(rng, ns, rad=(0.005, 0.05))
    tx, ty, _, tr = particles(rng, nt, rad=(0.005, 0.05))
    u, v = pair_sum([T(a) for a in src], [T(tx), T(ty)], T(tr), core)
    at = np.arange(0, nt, 100)
    ref = O.points_on_points(core, *src, tx[at], ty[at], tr[at])
    assert rel_l2(np.concatenate([u.cpu().numpy()[at], v.cpu().numpy()[at]]), np.concatenate(ref)) <= 1e-12
