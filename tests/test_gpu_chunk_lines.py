"""The sum over chunks on both sides of the targets from which a thread takes one of them whatever the
chunks (65,536), in two components and three, adding to what is there, against the oracle on a sample."""
import numpy as np
import pytest
import torch

import oracle as O
from helpers import circle_panels, particles, rel_l2
from omega2d_amd import device as dv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nt", [65535, 65536, 65537])
def test_many_targets_and_chunks(nt):
    rng = np.random.default_rng(nt)
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    tx, ty = rng.uniform(0.6, 3, nt), rng.uniform(-2, 2, nt)
    at = np.arange(0, nt, 61)
    base = [rng.normal(size=nt) for _ in range(3)]
    nx, ny, idx = circle_panels(100)  # a thread or a wave takes a panel chunk: 32 chunks here
    nx, ny = nx.astype(np.float64), ny.astype(np.float64)
    vs, ss = rng.normal(size=100), rng.normal(size=100)
    got = dv.panels_on_points(T(nx), T(ny), T(idx.astype(np.int32)), T(vs), T(ss), T(tx), T(ty),
                              tu=T(base[0]), tv=T(base[1]))
    for g, b, r in zip(got, base, O.panels_on_points(nx, ny, idx, vs, ss, tx[at], ty[at])):
        assert rel_l2(g.cpu().numpy()[at], b[at] + r) <= 1e-12
    sx, sy, s, r = particles(rng, 3000)
    got = dv.points_on_points(T(sx), T(sy), T(s), T(r), T(tx), T(ty), core="rm", results="vort",
                              tu=T(base[0]), tv=T(base[1]), aux=T(base[2]))
    for g, b, e in zip(got, base, O.points_on_points("rm", sx, sy, s, r, tx[at], ty[at], None, "vort")):
        assert rel_l2(g.cpu().numpy()[at], b[at] + e) <= 1e-12
