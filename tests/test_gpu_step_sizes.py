"""The vector work of a step takes one count for all of its arrays: arrays of other sizes are refused
before anything is launched."""
import pytest
import torch

from omega2d_amd import device as dv

pytestmark = pytest.mark.gpu


def Z(*n):
    return [torch.zeros(k, dtype=torch.float64, device="cuda") for k in n]


def one(k=1):
    return Z(k)[0]


CALLS = [
    lambda: dv.rk_advance(*Z(4, 3), Z(4), Z(4), [1.0], 0.1),
    lambda: dv.rk_advance(*Z(4, 4), Z(3), Z(4), [1.0], 0.1),
    lambda: dv.rk_advance(*Z(4, 4), Z(4, 4), Z(4, 3), [0.5, 0.5], 0.1),
    lambda: dv.rk_advance(*Z(4, 4), Z(4, 4), Z(4, 4), [1.0], 0.1),
    lambda: dv.rk_advance(*Z(4, 4), Z(4), Z(4), [1.0], 0.1, *Z(4, 5)),
    lambda: dv.finalize(*Z(4, 3), (0.0, 0.0), 1.0),
    lambda: dv.body_rhs(*Z(4, 4), (0.0, 0.0), 1.0, *Z(4, 4, 4, 3), 2, one(), 1.0, one()),
    lambda: dv.body_rhs(*Z(4, 4), (0.0, 0.0), 1.0, *Z(4, 4, 4, 4), 2, one(), 1.0, one(0)),
    lambda: dv.body_unpack(one(4), 2),
    lambda: dv.body_unpack(one(0), 1),
    lambda: dv.body_strengths(*Z(4, 4), one(), *Z(4, 4, 4, 3)),
    lambda: dv.body_strengths(*Z(4, 4), one(0), *Z(4, 4, 4, 4)),
]


@pytest.mark.parametrize("k", range(len(CALLS)))
def test_other_sizes_are_refused(k):
    with pytest.raises(ValueError):
        CALLS[k]()
