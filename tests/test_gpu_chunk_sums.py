"""The sum over source or target chunks, with a thread per target (below 8 chunks) and with 16 waves
per 64 targets, for two, three and four components: adding to what is there, at the edges of 64 targets
and of the waves' shares, against the oracle at the fp64 form's 1e-12 relative L2."""
import numpy as np
import pytest
import torch

import oracle as O
from helpers import particles, rel_l2
from omega2d_amd import device as dv

pytestmark = pytest.mark.gpu


def T(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("results", ["vel", "vort"])
@pytest.mark.parametrize("ns", [1, 65, 449, 513, 577, 2000])
@pytest.mark.parametrize("nt", [1, 63, 64, 65, 130])
def test_velocity_chunks(ns, nt, results):
    rng = np.random.default_rng(ns + nt)
    sx, sy, ss, sr = particles(rng, ns, rad=(0.05, 0.3))
    tx, ty, _, _ = particles(rng, nt)
    out = [rng.normal(size=nt) for _ in range(3 if results == "vort" else 2)]
    dev = [T(o) for o in out]
    dv.points_on_points(T(sx), T(sy), T(ss), T(sr), T(tx), T(ty), core="rm", results=results,
                        tu=dev[0], tv=dev[1], aux=dev[2] if results == "vort" else None)
    ref = O.points_on_points("rm", sx, sy, ss, sr, tx, ty, None, results)
    for d, o, r in zip(dev, out, ref):
        assert rel_l2(d.cpu().numpy(), o + r) <= 1e-12


@pytest.mark.parametrize("ns", [1, 65, 1000])
@pytest.mark.parametrize("nt", [200, 257, 1793, 2049, 4097])
def test_adjoint_chunks(ns, nt):
    rng = np.random.default_rng(ns + nt)
    sx, sy, ss, sr = particles(rng, ns, rad=(0.05, 0.3))
    tx, ty, gu, _ = particles(rng, nt)
    gv = rng.normal(size=nt)
    out = [rng.normal(size=ns) for _ in range(4)]
    dev = [T(o) for o in out]
    dv.points_on_points_adjoint(T(sx), T(sy), T(ss), T(sr), T(tx), T(ty), T(gu), T(gv), core="rm",
                                out=dev)
    ref = O.points_on_points_adjoint("rm", sx, sy, ss, sr, tx, ty, gu, gv)
    for d, o, r in zip(dev, out, ref):
        assert rel_l2(d.cpu().numpy(), o + r) <= 1e-12
