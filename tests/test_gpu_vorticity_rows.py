"""The vorticity sum at the lines where its source tiles are shared by one, two and three rows of
workgroups (8,192, 16,384 and 24,576 sources on enough targets to fill the chip), at radii that reach a
few boxes and all of them, against the oracle on a sample: 1e-12 relative L2."""
import numpy as np
import pytest
import torch

import oracle as O
from helpers import rel_l2
from omega2d_amd import device as dv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("radius", [0.004, 2.0])
@pytest.mark.parametrize("ns", [1, 257, 8191, 8193, 16384, 16385, 24577])
def test_rows(ns, radius):
    rng = np.random.default_rng(ns)
    nt = 99999
    sx, sy = rng.uniform(-1, 1, ns), rng.uniform(-1, 1, ns)
    ss, sr = rng.normal(size=ns), np.full(ns, radius)
    tx, ty, tw = rng.uniform(-1, 1, nt), rng.uniform(-1, 1, nt), rng.normal(size=nt)
    T = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    got = dv.points_vorticity(T(sx), T(sy), T(ss), T(sr), T(tx), T(ty), tw=T(tw)).cpu().numpy()
    at = np.arange(0, nt, 50)
    ref = tw[at] + O.points_vorticity(sx, sy, ss, sr, tx[at], ty[at])
    assert rel_l2(got[at], ref) <= 1e-12
