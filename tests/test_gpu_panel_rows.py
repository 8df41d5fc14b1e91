"""The clustered panel sums at the edges of their rows of clusters (dealt out over the rows, 16 to LDS
at a time), partial clusters and waves, and of the particle chunks whose far sums each wave reduces by
exchanges, against the oracle: 1e-12 relative L2, the panel sums' own bar."""
import numpy as np
import pytest

import oracle as O
import omega2d_amd as o2d
from helpers import circle_panels, rel_l2

pytestmark = pytest.mark.gpu


def around(rng, n):
    r = np.where(rng.uniform(size=n) < 0.5, 0.5 * rng.uniform(1.001, 1.1, n), rng.uniform(0.6, 3, n))
    th = rng.uniform(0, 2 * np.pi, n)
    return r * np.cos(th), r * np.sin(th)


@pytest.mark.parametrize("npan", [128, 129, 545, 1031, 2048])
@pytest.mark.parametrize("n", [1, 63, 65, 257, 1023, 1024, 1025, 20011])
def test_panel_sums_match_oracle(npan, n):
    rng = np.random.default_rng(npan + n)
    nx, ny, idx = circle_panels(npan)
    nx, ny = nx.astype(np.float64), ny.astype(np.float64)
    x, y = around(rng, n)
    s, vs, ss = rng.normal(size=n), rng.normal(size=npan), rng.normal(size=npan)
    for sheet in (None, ss):
        for g, r in zip(o2d.panels_on_points(nx, ny, idx, vs, sheet, x, y),
                        O.panels_on_points(nx, ny, idx, vs, sheet, x, y)):
            assert rel_l2(g, r) <= 1e-12
    for g, r in zip(o2d.points_on_panels(x, y, s, nx, ny, idx),
                    O.points_on_panels(x, y, s, nx, ny, idx)):
        assert rel_l2(g, r) <= 1e-12


def test_more_targets_than_rows_to_share():
    # one row: every cluster passes through LDS in stages, sums added to the outputs directly
    rng = np.random.default_rng(3)
    nx, ny, idx = circle_panels(600)
    nx, ny, vs = nx.astype(np.float64), ny.astype(np.float64), rng.normal(size=600)
    x, y = around(rng, 1 << 20)
    got = o2d.panels_on_points(nx, ny, idx, vs, None, x, y)
    at = rng.integers(0, len(x), 3000)
    for g, r in zip(got, O.panels_on_points(nx, ny, idx, vs, None, x[at], y[at])):
        assert rel_l2(g[at], r) <= 1e-12
