"""Neighbour search at the edges of its paths: one-workgroup binning up to 4,000 points and
the general one beyond, every length of the register list, queries that are or are not the
data, clouds away from the origin, repeated points. Compared with brute force, order included
(ties by lower index)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,n,k", [(2, 65, 64), (1, 4000, 7), (2, 4000, 16), (2, 4001, 17), (3, 3999, 21),
                                     (3, 4001, 25), (3, 5000, 33), (2, 5000, 41), (3, 4500, 49), (1, 4500, 64),
                                     (2, 2, 2), (3, 1, 1), (2, 700, 1)])
def test_knn_paths_match_bruteforce(RBF, O, gpu, dim, n, k):
    rng = np.random.default_rng(n + k)
    pts = rng.random((n, dim)) ** 2 + np.array([3.0e3, -2.0, 0.0])[:dim]
    pts[n // 2:n // 2 + 3] = pts[:1]  # repeated points
    assert np.array_equal(RBF.find_neighbors(pts, k=k), O.knn(pts, pts, k))
    q = pts[rng.integers(0, n, 777)] + rng.normal(0, 0.3, (777, dim))
    assert np.array_equal(RBF.find_neighbors(pts, q, k=k), O.knn(pts, q, k))


@pytest.mark.parametrize("dim,n,nq", [(1, 70_001, 0), (2, 70_001, 0), (3, 70_001, 0), (2, 300, 66_000)])
def test_knn_order_is_a_spatial_permutation(RBF, gpu, dim, n, nq):
    """The processing order that comes with the search: a permutation of the queries whose
    consecutive entries lie near each other (within a few cells on average)."""
    import torch

    rng = np.random.default_rng(dim)
    x = torch.as_tensor(rng.random((n, dim)), device=gpu)
    q = x if nq == 0 else torch.as_tensor(rng.random((nq, dim)), device=gpu)
    adj, order = RBF._lib.knn(x, q, 5, order=True)
    assert torch.equal(adj, RBF._lib.knn(x, q, 5))
    o = order.long()
    assert torch.equal(torch.sort(o)[0], torch.arange(q.shape[0], device=gpu))
    step = (q[o[1:]] - q[o[:-1]]).norm(dim=1).mean().item()
    assert step < 8.0 * n ** (-1.0 / dim), step


def test_operator_with_and_without_order_agree(RBF, gpu):
    """70,000 points: weights of the ordered build equal the unordered ones bit for bit."""
    import torch

    pts = torch.as_tensor(np.random.default_rng(2).random((70_000, 2)), device=gpu)
    op = RBF.gradient(pts, k=14)
    assert op._row_order is not None
    w = op.vals.clone()
    op._row_order, op.SPATIAL_ORDER_MIN = None, 10 ** 12
    op.update_weights()
    assert torch.equal(op.vals, w)
