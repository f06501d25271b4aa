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


@pytest.mark.parametrize("dim,k", [(1, 5), (1, 32), (2, 1), (2, 16), (2, 20), (2, 32), (3, 17), (3, 24), (2, 64)])
def test_knn_wavefront_and_lane_per_query_agree(RBF, gpu, dim, k):
    """Many queries at once (a lane each, up to k = 32) against the same queries in parts (a
    wavefront each): a cloud with clusters, a lattice of ties, repeated points, far queries,
    ragged lists."""
    import torch

    rng = np.random.default_rng(100 * dim + k)
    x = np.concatenate([rng.random((3000, dim)), 0.5 + 1e-3 * rng.standard_normal((1500, dim)),
                        rng.integers(0, 12, (1500, dim)) / 11.0])
    n = 264_000 if dim == 3 else 66_000
    q = np.concatenate([x, x[rng.integers(0, 6000, n - 6010)] + rng.normal(0, 0.05, (n - 6010, dim)),
                        rng.normal(0, 30.0, (10, dim))])
    x, q = torch.as_tensor(x, device=gpu), torch.as_tensor(q, device=gpu)
    whole = RBF._lib.knn(x, q, k)
    part = n // 11
    parts = torch.cat([RBF._lib.knn(x, q[a:a + part].contiguous(), k) for a in range(0, n, part)])
    assert torch.equal(whole, parts)
    for m in (part, n):
        c = torch.as_tensor(rng.integers(0, k + 1, m), device=gpu)
        ptr = torch.cat([torch.zeros(1, dtype=torch.int64, device=gpu), torch.cumsum(c, 0)])
        ragged = RBF._lib.knn(x, q[:m].contiguous(), k, q_ptr=ptr)
        mask = torch.arange(k, device=gpu)[None, :] < c[:, None]
        assert torch.equal(ragged, whole[:m][mask])


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


@pytest.mark.parametrize("dim,k", [(1, 9), (2, 12), (2, 40), (3, 20), (3, 33)])
def test_knn_inside_dense_clusters(RBF, O, gpu, dim, k):
    """Clusters of a hundred to ten thousand times the mean density, where the block of two rings
    holds thousands of points and both searches go ring by ring from the query's own cell:
    against brute force, in the clusters, at their rims and between them."""
    import torch

    rng = np.random.default_rng(10 * dim + k)
    x = np.concatenate([0.5 + 0.02 * rng.standard_normal((9000, dim)), 0.2 + 2e-4 * rng.standard_normal((6000, dim)),
                        rng.random((1000, dim))])
    x = x[rng.permutation(len(x))]
    some = np.concatenate([x[:1500], 0.5 + 0.06 * rng.standard_normal((500, dim)), 0.2 + 6e-4 * rng.standard_normal((500, dim))])
    want = O.knn(x, some, k)
    assert np.array_equal(RBF.find_neighbors(x, some, k=k), want)
    if k <= 32:  # the same queries among enough others that a lane takes each
        n = 263_000 if dim == 3 else 66_000
        q = torch.as_tensor(np.concatenate([some, x[rng.integers(0, len(x), n)]]), device=gpu)
        got = RBF._lib.knn(torch.as_tensor(x, device=gpu), q, k)
        assert np.array_equal(got[:len(some)].cpu().numpy(), want)


@pytest.mark.parametrize("dim,n", [(2, 4000), (3, 512), (3, 513), (3, 4000)])
def test_knn_many_queries_of_a_small_cloud(RBF, O, gpu, dim, n):
    """More queries than wavefronts take, not the points themselves, of clouds small enough for
    one workgroup's binning: in 3-D beyond 512 points the queries are binned too."""
    import torch

    rng = np.random.default_rng(n)
    x, some = rng.random((n, dim)), rng.random((1000, dim)) * 1.4 - 0.2
    q = torch.as_tensor(np.concatenate([some, rng.random((265_000, dim))]), device=gpu)
    got = RBF._lib.knn(torch.as_tensor(x, device=gpu), q, 20)
    assert np.array_equal(got[:1000].cpu().numpy(), O.knn(x, some, 20))
    part = RBF._lib.knn(torch.as_tensor(x, device=gpu), q[-50_000:].contiguous(), 20)  # (a wavefront each)
    assert torch.equal(got[-50_000:], part)
