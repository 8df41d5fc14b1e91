"""Calls on host arrays whose arrays travel packed (up to 16 MiB) or one by one, against the device
entry on the same values: the same sums bit for bit, rounded to float in the float entry. Arrays that
are the sources' own, in part or whole, inert targets, results that add to what is there, and sizes at
the ends of an array's 32-element padding and on both sides of the limit."""
import numpy as np
import pytest
import torch

import omega2d_amd as o2d
from omega2d_amd import device as dv

pytestmark = pytest.mark.gpu


def both(dt, src, tgt, tr, results, out):
    """The host entry's results, and the device entry's on the same values."""
    got = [o.copy() for o in out]
    kw = dict(core="v2", precision="fp64", results=results)
    o2d.points_on_points(*src, *tgt, tr, tu=got[0], tv=got[1],
                         **(dict(aux=got[2]) if results != "vel" else {}), **kw)
    seen = {}  # the same host array is the same device array
    T = lambda a: None if a is None else seen.setdefault(  # noqa: E731
        id(a), torch.from_numpy(a.astype(np.float64)).cuda())
    ref = [torch.from_numpy(o.astype(np.float64)).cuda() for o in out]
    dv.points_on_points(*[T(a) for a in src], *[T(a) for a in tgt], T(tr), tu=ref[0], tv=ref[1],
                        aux=ref[2] if results != "vel" else None, **kw)
    return got, [r.cpu().numpy().astype(dt) for r in ref]


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("results", ["vel", "vort", "shear"])
@pytest.mark.parametrize("targets", ["self", "inert self", "x only", "y and radius", "other", "inert"])
@pytest.mark.parametrize("n", [1, 31, 32, 33, 1531])
def test_packed_arrays(n, targets, results, dt):
    rng = np.random.default_rng(n)
    new = lambda m: rng.uniform(0.1, 1.0, m).astype(dt)  # noqa: E731
    src = [new(n) for _ in range(4)]
    nt = n if targets not in ("other", "inert") else 2 * n + 3
    tgt, tr = {"self": (src[:2], src[3]), "inert self": (src[:2], None),
               "x only": ([src[0], new(nt)], new(nt)), "y and radius": ([new(nt), src[1]], src[3]),
               "other": ([new(nt), new(nt)], new(nt)), "inert": ([new(nt), new(nt)], None)}[targets]
    out = [rng.normal(size=nt).astype(dt) for _ in range(3)]
    got, ref = both(dt, src, tgt, tr, results, out)
    for g, r in zip(got[:2] if results == "vel" else got, ref):
        assert np.array_equal(g, r)


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("over", [False, True])
def test_both_sides_of_the_limit(over, dt):
    n = (16 << 20) // (4 * np.dtype(dt).itemsize) - (0 if over else 64)
    rng = np.random.default_rng(1)
    src = [rng.uniform(0.1, 1.0, n).astype(dt) for _ in range(4)]
    tgt = [rng.uniform(0.1, 1.0, 3).astype(dt) for _ in range(2)]
    got, ref = both(dt, src, tgt, None, "vel", [np.zeros(3, dt)] * 3)
    assert np.array_equal(got[0], ref[0]) and np.array_equal(got[1], ref[1])
