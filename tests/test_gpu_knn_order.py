"""The processing order that comes with a search of few queries in a much larger cloud (most
of whose cells hold none of them): a permutation, and the same neighbours."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,n,nq", [(1, 70_001, 63), (2, 300_000, 1), (2, 70_001, 700), (2, 200_000, 30_000),
                                      (3, 70_001, 65), (3, 200_000, 5_000), (3, 300_000, 40_001)])
def test_order_of_few_queries_is_a_permutation(RBF, gpu, dim, n, nq):
    import torch

    rng = np.random.default_rng(nq)
    x = torch.as_tensor(rng.random((n, dim)), device=gpu)
    q = torch.as_tensor(rng.random((nq, dim)) * 1.5 - 0.25, device=gpu)  # (some outside the cloud)
    adj, order = RBF._lib.knn(x, q, 7, order=True)
    assert torch.equal(adj, RBF._lib.knn(x, q, 7))
    assert torch.equal(torch.sort(order.long())[0], torch.arange(nq, device=gpu))
