"""Calls on host arrays on both sides of the outputs' limit for travelling packed (3 MiB), against the
device entry on the same values, bit for bit."""
import numpy as np
import pytest

from test_gpu_packed_host import both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("results", ["vel", "vort"])
@pytest.mark.parametrize("over", [False, True])
def test_both_sides_of_the_outputs_limit(over, results, dt):
    outs = 2 if results == "vel" else 3
    nt = (3 << 20) // (outs * np.dtype(dt).itemsize) // 32 * 32 + (1 if over else 0)
    rng = np.random.default_rng(outs)
    src = [rng.uniform(0.1, 1.0, 50).astype(dt) for _ in range(4)]
    tgt = [rng.uniform(0.1, 1.0, nt).astype(dt) for _ in range(2)]
    out = [rng.normal(size=nt).astype(dt) for _ in range(3)]
    got, ref = both(dt, src, tgt, None, results, out)
    for g, r in zip(got[:outs], ref):
        assert np.array_equal(g, r)
