"""The treecode's error at every order against that of the plain scheme its order is defined by, made
here in numpy: Morton leaves of 64 sources, four cells to a parent, a cell acting on 64 Morton-ordered
targets through its first `order` moments when its radius is at most theta times its distance from each of
them, and pair by pair sums of the leaves that are left. The error may be no larger than the plain
scheme's: groups, local expansions and orders left out must not add to it."""
import numpy as np
import pytest
import torch

import oracle as O
from omega2d_amd import device as dv

pytestmark = pytest.mark.gpu

LEAF, FAN, GROUP = 64, 4, 64
OPTIONS = [(0.6, 28), (0.5, 20), (0.6, 16), (0.6, 8), (0.6, 4), (0.6, 2), (0.6, 1), (0.8, 16), (0.9, 8),
           (0.9, 32), (0.3, 6), (0.3, 3), (0.3, 1), (0.1, 3)]


def curve(z):
    x, y = z.real, z.imag
    ext = max(np.ptp(x), np.ptp(y))
    return np.argsort(O.morton_keys(x, y, x.min(), y.min(), 1.0 / ext), kind="stable")


class Plain:
    def __init__(self, z, q, t):
        o = curve(z)
        self.z, self.q = z[o], q[o]
        self.torder = curve(t)
        self.t = t[self.torder].reshape(-1, GROUP)
        self.levels, size = [], LEAF
        while True:
            cells = []
            for a in range(0, len(z), size):
                p = self.z[a:a + size]
                c = complex((p.real.min() + p.real.max()) / 2, (p.imag.min() + p.imag.max()) / 2)
                cells.append((a, min(a + size, len(z)), c, np.abs(p - c).max()))
            self.levels.append(cells)
            if len(cells) == 1:
                break
            size *= FAN

    def sum(self, theta, order):
        """sum_j q_j / (t - z_j), in the targets' input order"""
        out = np.zeros(self.t.shape, complex)
        alive = np.ones((1, len(self.t)), bool)  # of each cell: the groups that open it
        for level in reversed(range(len(self.levels))):
            cells = self.levels[level]
            opened = np.zeros((len(cells), len(self.t)), bool)
            for i, (a, b, c, r) in enumerate(cells):
                g = np.flatnonzero(alive[i])
                d = self.t[g] - c
                far = (r <= theta * np.abs(d)).all(1)
                f, n = g[far], g[~far]
                if len(f):
                    w, m = 1.0 / d[far], self.z[a:b] - c
                    acc = np.zeros(w.shape, complex)
                    for k in reversed(range(order)):
                        acc = acc * w + (self.q[a:b] * m**k).sum()
                    out[f] += acc * w
                if level == 0:
                    for k in n:
                        e = self.t[k][:, None] - self.z[a:b]
                        out[k] += np.where(e == 0, 0, self.q[a:b] / np.where(e == 0, 1, e)).sum(1)
                else:
                    opened[i, n] = True
            alive = np.repeat(opened, FAN, 0)
        res = np.empty(out.size, complex)
        res[self.torder] = out.ravel()
        return res


@pytest.mark.parametrize("nt", [0, 2048])  # the sources themselves, or targets a quarter as dense
@pytest.mark.parametrize("kind", ["square", "line"])
def test_error_is_within_the_plain_schemes(kind, nt):
    rng = np.random.default_rng(nt + len(kind))
    ns = 16384
    draw = lambda n: (rng.uniform(-1, 1, n) + 1j * (  # noqa: E731
        rng.uniform(-1, 1, n) if kind == "square" else 0.01 * rng.normal(size=n)))
    z, q = draw(ns), rng.normal(0.3, 1.0, ns)
    t = draw(nt) if nt else z
    r = np.full(ns, 1e-9)  # pairs are 1/d^2: the plain scheme has no cores
    ref = O.points_on_points("gauss", z.real, z.imag, q, r, t.real, t.imag)
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    d = [T(z.real), T(z.imag), T(q), T(r)]
    td = [T(t.real), T(t.imag)] if nt else d[:2]
    plain = Plain(z, q, t)
    # u - i v = -i S: S = v + i u
    error = lambda u, v: np.sqrt(np.sum((u - ref[0])**2 + (v - ref[1])**2))  # noqa: E731
    for theta, order in OPTIONS:
        s = plain.sum(theta, order)
        got = [g.cpu().numpy() for g in dv.points_on_points_tree(*d, *td, core="gauss", theta=theta,
                                                                 order=order)]
        mine, its = error(*got), error(s.imag, s.real)
        print(kind, nt, theta, order, "%.2e %.2f" % (its, mine / its))
        assert mine <= its, (theta, order, mine / its)
