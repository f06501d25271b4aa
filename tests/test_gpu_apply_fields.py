"""Many-field applies staged through LDS: byte offsets into an X of up to 4 GB against the
general addressing (taken where the number of points of X is not given), at row lengths around
the six entries a lane has in flight, both layouts of the fields, several value arrays."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k,F,op", [(6, 8, "d1"), (7, 8, "grad"), (12, 9, "d1"), (13, 16, "d1"), (17, 17, "grad"),
                                    (20, 64, "d1"), (30, 33, "d1"), (5, 16, "grad")])
@pytest.mark.parametrize("ragged", [False, True])
def test_near_addressing_equals_general(RBF, O, gpu, k, F, op, ragged):
    import torch

    rng = np.random.default_rng(k * F)
    pts = rng.random((1237, 2))
    adj = O.knn(pts, pts, k)
    if ragged:
        adj = [a[:max(5, k - i % 3)] for i, a in enumerate(adj)]
    L = RBF.Partial(1, 1) if op == "d1" else RBF.Jacobian(2)
    W = RBF.RadialBasisOperator(L, pts, basis=RBF.PHS(3, poly_deg=1), adjl=adj)
    X = torch.as_tensor(rng.standard_normal((1237, F)), device=gpu)
    for x in (X, X.t().contiguous().t()):  # point-major and field-major
        s, y = W._spmv_args(x)
        s.mapping = 2
        RBF._lib.spmv(s, W.dev)
        near = y.clone()
        s.n_cols = 0
        y.zero_()
        RBF._lib.spmv(s, W.dev)
        assert torch.equal(near, y)
        ref = W.weights()
        ref = ref if isinstance(ref, tuple) else (ref,)
        for c, m in enumerate(ref):
            e = m @ x.cpu().numpy()
            scale = (abs(m) @ np.abs(x.cpu().numpy())).max()  # (k products, summed either way)
            assert np.abs(near[c].cpu().numpy() - e).max() <= 64 * 2.0 ** -53 * scale
