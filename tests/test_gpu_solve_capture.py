"""Solves captured into a graph after some eager ones with the same factors, at every point of the way
from the factors to the inverse: the capture is taken (no allocation, no library call), and its replays
stay right when later eager solves build the inverse between them. Against LAPACK; the matrices and the
bar are those of the solves without a graph."""
import numpy as np
import pytest
import torch

from helpers import rel_l2
from omega2d_amd import device as dv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("before", [0, 1, 2, 3, 4, 5])
@pytest.mark.parametrize("n", [1, 64, 65, 256, 257, 513])
def test_captured_solves(n, before):
    rng = np.random.default_rng(n + before)
    A = (np.eye(n) + 0.25 * rng.normal(size=(n, n)) / np.sqrt(n))[rng.permutation(n)]
    dv.bem_factor(torch.from_numpy(np.ascontiguousarray(A.T)).cuda())

    def eager():
        b = rng.normal(size=n)
        x = dv.bem_solve(torch.from_numpy(b).cuda())
        assert rel_l2(x.cpu().numpy(), np.linalg.solve(A, b)) <= 1e-12

    for _ in range(before):
        eager()
    b1, b2 = (torch.zeros(n, dtype=torch.float64, device="cuda") for _ in range(2))
    x1, x2 = torch.empty_like(b1), torch.empty_like(b1)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        dv.bem_solve(b1, x1)
        dv.bem_solve(b2, x2)
    for _ in range(6):
        h1, h2 = rng.normal(size=n), rng.normal(size=n)
        b1.copy_(torch.from_numpy(h1))
        b2.copy_(torch.from_numpy(h2))
        graph.replay()
        torch.cuda.synchronize()
        assert rel_l2(x1.cpu().numpy(), np.linalg.solve(A, h1)) <= 1e-12
        assert rel_l2(x2.cpu().numpy(), np.linalg.solve(A, h2)) <= 1e-12
        eager()


def test_solves_past_the_blocked_factorisation():
    """From order 6,145 the factors are the library's: three solves by them, the later ones by the
    inverse, and a captured one."""
    n = 6145
    g = torch.Generator(device="cuda").manual_seed(1)
    A = torch.randn((n, n), dtype=torch.float64, device="cuda", generator=g) * (0.25 / np.sqrt(n))
    A += torch.eye(n, dtype=torch.float64, device="cuda")
    A = A[torch.randperm(n, device="cuda", generator=g)]
    dv.bem_factor(A.T.contiguous())
    new = lambda: torch.randn(n, dtype=torch.float64, device="cuda", generator=g)  # noqa: E731

    def check(x, b):
        assert float((A @ x - b).norm() / b.norm()) <= 1e-12

    b = new()
    check(dv.bem_solve(b), b)
    held, x = new(), torch.empty_like(b)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        dv.bem_solve(held, x)
    for _ in range(4):
        held.copy_(new())
        graph.replay()
        torch.cuda.synchronize()
        check(x, held)
        b = new()
        check(dv.bem_solve(b), b)


@pytest.mark.parametrize("n", [16, 17, 63, 64, 65, 255, 256, 257])
def test_solves_in_place(n):
    """Every solve of a run in place: by the factors, then by the inverse on both sides of the order up to
    which its product is one launch."""
    rng = np.random.default_rng(n)
    A = (np.eye(n) + 0.25 * rng.normal(size=(n, n)) / np.sqrt(n))[rng.permutation(n)]
    dv.bem_factor(torch.from_numpy(np.ascontiguousarray(A.T)).cuda())
    for k in range(6):
        b = rng.normal(size=n)
        x = torch.from_numpy(b).cuda()
        dv.bem_solve(x, x)
        assert rel_l2(x.cpu().numpy(), np.linalg.solve(A, b)) <= 1e-12, k
