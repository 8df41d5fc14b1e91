"""Repeated solves with one factorisation against LAPACK, at the edges of the 64-row blocks: the
first three by block substitution, the fourth builds the inverse and multiplies by it, in place
and not. The matrices are well conditioned (I + 1/4 of a random matrix of spectral radius about
1), so the bar is the fp64 form's 1e-12."""
import numpy as np
import pytest
import torch

from helpers import rel_l2
from omega2d_amd import device as dv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 127, 129, 513, 1985, 2049])
def test_repeated_solves_match_lapack(n):
    rng = np.random.default_rng(n)
    A = (np.eye(n) + 0.25 * rng.normal(size=(n, n)) / np.sqrt(n))[rng.permutation(n)]
    dv.bem_factor(torch.from_numpy(np.ascontiguousarray(A.T)).cuda())
    for k in range(6):
        b = rng.normal(size=n)
        db = torch.from_numpy(b).cuda()
        x = dv.bem_solve(db, db) if k % 2 else dv.bem_solve(db)
        assert rel_l2(x.cpu().numpy(), np.linalg.solve(A, b)) <= 1e-12, k
