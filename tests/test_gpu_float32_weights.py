"""Operators of single-precision points round their weights to FP32, so their builds keep to
the kernels whose weights they have always had: the FP64 weights of the null-space
elimination (kernel 8) differ from those by some units of the last place, which moves an FP32
rounding here and there. Every weight here is the FP32 rounding of the FP64 build of the
same points on the kernel that the single-precision build names."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
K_NSE = 8


def _pinned_build(RBF, kernels, plan, build):
    for b, k in enumerate(kernels):
        if k >= 0:
            RBF._lib.tune_bucket(b, k)
    RBF._lib.tune_plan(plan)
    try:
        return build()
    finally:
        RBF._lib.tune_plan(0)
        for b in range(3):
            RBF._lib.tune_bucket(b, -1)


@pytest.mark.parametrize("dim,kind,deg,k,op,n,kernel",
                         [(2, 3, 2, 12, "laplacian", 900, 6), (2, 5, 3, 20, "hessian", 1001, 0),
                          (2, 5, 3, 20, "hessian", 9001, 0), (2, 7, 3, 20, "hessian", 9001, 7),
                          (2, 3, 3, 27, "laplacian", 3000, 5), (2, 3, 3, 27, "laplacian", 5000, 5),
                          (3, 3, 2, 20, "gradient", 5001, 7), (3, 3, 2, 20, "laplacian", 5001, 7),
                          (3, 5, 3, 40, "gradient", 700, 7)])
def test_uniform_builds_keep_their_kernels(RBF, gpu, dim, kind, deg, k, op, n, kernel):
    import torch

    pts = torch.as_tensor(np.random.default_rng(n).random((n, dim)), device=gpu).float()
    L = {"laplacian": RBF.Laplacian, "gradient": lambda: RBF.Jacobian(dim), "hessian": lambda: RBF.Hessian(dim)}[op]()
    basis = RBF.PHS(kind, poly_deg=deg)
    RBF._lib.tune_reset()
    RBF.RadialBasisOperator(L, pts.double(), basis=basis, k=k)  # (what it may leave in the tuning map)
    w = RBF.RadialBasisOperator(L, pts, basis=basis, k=k)
    kern = RBF._lib.last_build_buckets()[1]
    assert [x for x in kern if x >= 0] == [kernel]
    ref = _pinned_build(RBF, kern, 0, lambda: RBF.RadialBasisOperator(L, pts.double(), basis=basis, k=k))
    assert RBF._lib.last_build_buckets()[1] == kern
    assert torch.equal(w.vals, ref.vals.float().double())
    f = torch.sin(3.0 * pts[:, 0])
    first = w.vals.clone()
    g = w.capture(f)
    for _ in range(3):
        w.vals.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(w.vals, first)


def test_uneven_build_runs_no_null_space_class(RBF, gpu):
    import torch

    rng = np.random.default_rng(4)
    pts = torch.as_tensor(rng.random((2000, 2)), device=gpu).float()
    idx = RBF._lib.knn(pts.double(), pts.double(), 50).cpu().numpy()
    adjl = [idx[i, :kk] for i, kk in enumerate(rng.integers(12, 51, 2000))]
    basis = RBF.PHS(3, poly_deg=2)
    ref = _pinned_build(RBF, (-1, -1, -1), 1, lambda: RBF.laplacian(pts.double(), basis=basis, adjl=adjl))
    RBF.laplacian(pts.double(), basis=basis, adjl=adjl)
    assert RBF._lib.last_build_stats()[3] > 1000  # (the classes take most of the FP64 build)
    w = RBF.laplacian(pts, basis=basis, adjl=adjl)
    assert RBF._lib.last_build_stats()[3] == 0
    assert torch.equal(w.vals, ref.vals.float().double())
