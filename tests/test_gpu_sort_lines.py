"""The device key sort on both sides of the line between its tiles of 8,192 keys and the library sort,
bit-exact against numpy's stable argsort."""
import pytest

from test_gpu_sort import test_morton_order_is_the_stable_order as check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spread", ["wide", "clustered", "single"])
@pytest.mark.parametrize("n", [1048576, 2097151, 2097152, 2097153])
def test_both_sides_of_the_tiles(n, spread):
    check(n, spread)
