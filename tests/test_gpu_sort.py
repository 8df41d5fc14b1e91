"""The device key sort against numpy's stable argsort of the oracle's Morton keys, bit-exact, at
the edges of its ranges: ranks by comparison (to 12,288 keys, with 2, 4, 8 and 12 keys per thread,
16, 32 or 64 ranks per workgroup), the tiled passes with 2, 4, 8 and 16 keys per thread (from 12,289,
65,537, 262,145 and 1,048,577) and the library sort past 4,194,304 keys; spread keys, keys that
share their high digits, and one key throughout."""
import numpy as np
import pytest
import torch

import oracle as O
from omega2d_amd import device as dv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spread", ["wide", "clustered", "single"])
@pytest.mark.parametrize("n", [1, 15, 63, 65, 1024, 1025, 2048, 2049, 4096, 4097, 8191, 8192, 8193,
                               12287, 12288, 12289, 65536, 65537, 262145, 1048577,
                               4194305])
def test_morton_order_is_the_stable_order(n, spread):
    rng = np.random.default_rng(n)
    if spread == "wide":
        x, y = rng.uniform(-4, 4, n), rng.normal(0, 1.5, n)
    elif spread == "clustered":  # a few tight clusters with repeated positions
        c = rng.integers(0, 3, n)
        x = np.array([-3.0, 0.5, 0.5001])[c] + 1e-3 * np.round(rng.uniform(size=n), 2)
        y = np.array([2.0, -1.0, -1.0])[c] + 1e-3 * np.round(rng.uniform(size=n), 2)
    else:
        x, y = np.full(n, 0.25), np.full(n, -0.5)
    x0, y0, inv = -4.0, -8.0, 1.0 / 16.0
    keys, order = dv.morton_order(torch.from_numpy(x).cuda(), torch.from_numpy(y).cuda(), x0, y0,
                                  inv)
    torch.cuda.synchronize()
    ref = O.morton_keys(x, y, x0, y0, inv)
    want = np.argsort(ref, kind="stable").astype(np.uint32)
    assert np.array_equal(order.cpu().numpy().view(np.uint32), want)
    assert np.array_equal(keys.cpu().numpy().view(np.uint32), ref[want])
