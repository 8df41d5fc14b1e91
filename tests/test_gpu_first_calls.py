"""First calls of the clustered fp64 Gaussian sums: nothing is kept from a call before, and the pair by
pair sums behind the clusters need more room for partial sums than the clusters' shares, so the buffer
that both use moves within the call. The first call and the ones after it agree bit for bit, and with the
oracle at the fp64 form's 1e-12 relative L2."""
import numpy as np
import pytest
import torch

import oracle as O
from helpers import rel_l2
from omega2d_amd import _cabi, device as dv

pytestmark = pytest.mark.gpu


def T(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("kind,ns,nt", [("velocity", 300001, 3001), ("velocity", 60001, 9001),
                                        ("adjoint", 3001, 150001), ("adjoint", 20011, 20011)])
def test_first_call(kind, ns, nt, wide):
    rng = np.random.default_rng(ns + nt)
    x, y, tx, ty = (rng.uniform(-1, 1, n) for n in (ns, ns, nt, nt))
    s, r = rng.normal(size=ns), np.full(ns, 3.0 if wide else 0.002)
    gu, gv = rng.normal(size=nt), rng.normal(size=nt)
    n = ns if kind == "adjoint" else nt
    at = np.unique(np.linspace(0, n - 1, 60).astype(np.int64))
    if kind == "adjoint":
        args, call = (x, y, s, r, tx, ty, gu, gv), dv.points_on_points_adjoint
        ref = O.points_on_points_adjoint("gauss", x[at], y[at], s[at], r[at], tx, ty, gu, gv)
        kw = {}
    else:
        args, call = (x, y, s, r, tx, ty), dv.points_on_points
        ref = O.points_on_points("gauss", x, y, s, r, tx[at], ty[at], None)
        kw = dict(precision="fp64")
    args = [T(a) for a in args]
    if kind == "velocity":
        args.append(None)
    torch.cuda.synchronize()
    assert _cabi.lib().o2d_hip_release() == 0
    runs = [[g.cpu().numpy() for g in call(*args, core="gauss", **kw)] for _ in range(3)]
    for again in runs[1:]:
        assert all(np.array_equal(a, b) for a, b in zip(again, runs[0]))
    for g, e in zip(runs[0], ref):
        assert rel_l2(g[at], e) <= 1e-12
