"""GPU parity tests of the null-space elimination build (kernel id 8): every stencil against
the extended-precision oracle at max(1e-10, kappa_2(A) u), the bound the other kernels meet
(test_gpu_build.check_against_truth), at the edges of its shapes: one null point, the
last one of each slot and the first of the next, the largest; every column count; a number of
stencils that leaves the last wavefront part empty."""
import contextlib
from math import comb

import numpy as np
import pytest

from test_gpu_build import _op, check_against_truth

pytestmark = pytest.mark.gpu
K_NSE = 8


@contextlib.contextmanager
def pinned(RBF, kernel):
    for b in range(3):
        RBF._lib.tune_bucket(b, kernel)
    try:
        yield
    finally:
        for b in range(3):
            RBF._lib.tune_bucket(b, -1)


def _operator(RBF, O, dim, cols):
    A = O.abi
    d1 = [(c, A.OP_D1, c, 0, 1.0) for c in range(dim)]
    pairs = [(i, j) for i in range(dim) for j in range(i, dim)]
    table = {
        "lap": (RBF.Laplacian() + 0.5 * RBF.Partial(1, dim), 1, [(0, A.OP_LAP, 0, 0, 1.0), (0, A.OP_D1, dim - 1, 0, 0.5)]),
        "value": (RBF.Regrid(), 1, [(0, A.OP_VALUE, 0, 0, 1.0)]),
        "grad": (RBF.Jacobian(dim), dim, d1),
        "gradlap": (RBF.Stacked(RBF.Jacobian(dim), RBF.Laplacian()), dim + 1, d1 + [(dim, A.OP_LAP, 0, 0, 1.0)]),
        "two": (RBF.Stacked(RBF.MixedPartial(1, 2), RBF.Partial(2, 1)), 2,
                [(0, A.OP_MIXED, 0, 1, 1.0), (1, A.OP_D2, 0, 0, 1.0)]),
        "hess": (RBF.Hessian(dim), len(pairs), [(c, A.OP_D2 if i == j else A.OP_MIXED, i, j, 1.0)
                                               for c, (i, j) in enumerate(pairs)]),
    }
    return table[cols]


# (kind, dim, degree, null points k - m, operator)
CASES = [
    (3, 2, 1, 1, "grad"), (3, 2, 1, 3, "lap"), (3, 2, 1, 11, "grad"), (3, 2, 1, 12, "value"),
    (3, 2, 2, 1, "lap"), (3, 2, 2, 6, "lap"), (3, 2, 2, 9, "lap"), (3, 2, 2, 10, "lap"), (3, 2, 2, 14, "lap"),
    (3, 2, 2, 15, "lap"), (3, 2, 2, 16, "lap"), (3, 2, 2, 26, "lap"), (3, 2, 2, 7, "hess"), (3, 2, 2, 8, "grad"),
    (3, 2, 2, 13, "gradlap"), (3, 2, 2, 14, "gradlap"), (3, 2, 2, 14, "two"), (3, 2, 2, 26, "hess"),
    (5, 2, 2, 9, "value"), (5, 2, 3, 10, "hess"), (5, 2, 3, 13, "hess"), (5, 2, 3, 15, "lap"), (5, 2, 3, 20, "grad"),
    (3, 2, 3, 10, "lap"), (3, 2, 3, 16, "hess"), (3, 2, 4, 13, "hess"), (5, 2, 4, 15, "lap"), (5, 2, 4, 17, "grad"),
    (7, 2, 3, 12, "lap"), (7, 2, 4, 15, "lap"), (7, 2, 4, 16, "gradlap"),
    (3, 3, 1, 6, "grad"), (3, 3, 1, 9, "gradlap"), (3, 3, 1, 15, "lap"), (3, 3, 1, 10, "hess"), (3, 3, 1, 12, "two"),
    (3, 3, 2, 1, "lap"), (3, 3, 2, 10, "grad"), (3, 3, 2, 10, "hess"), (3, 3, 2, 13, "grad"), (3, 3, 2, 11, "hess"),
    (3, 3, 2, 15, "lap"), (3, 3, 2, 16, "lap"), (3, 3, 2, 25, "hess"), (5, 3, 2, 14, "gradlap"), (5, 3, 2, 26, "lap"),
    (5, 3, 3, 1, "lap"), (5, 3, 3, 16, "grad"), (5, 3, 3, 20, "gradlap"), (5, 3, 3, 20, "hess"),
    (5, 3, 3, 21, "gradlap"), (3, 3, 3, 26, "hess"), (3, 3, 3, 20, "lap"), (7, 3, 3, 19, "two"), (7, 3, 3, 26, "lap"),
]


@pytest.mark.parametrize("kind,dim,deg,nn,cols", CASES)
def test_nse_parity_against_truth(RBF, O, gpu, kind, dim, deg, nn, cols):
    """A random cloud with stencils one-sided at its faces; 401 stencils (not a multiple of 4)."""
    k = comb(dim + deg, dim) + nn
    pts = np.random.default_rng(100 * kind + 10 * deg + nn).random((401, dim))
    L, n_cols, terms = _operator(RBF, O, dim, cols)
    with pinned(RBF, K_NSE):
        op = RBF.RadialBasisOperator(L, pts, basis=RBF.PHS(kind, poly_deg=deg), k=k)
    _, kern = RBF._lib.last_build_buckets()
    assert K_NSE in kern, kern
    assert RBF._lib.last_build_stats()[0] <= len(pts) // 20  # breakdowns are rare for these pairings
    adj = op.adj_idx.cpu().numpy()
    check_against_truth(O, op.vals.cpu().numpy(), pts, pts, adj, O.basis_struct(kind, deg), _op(O, n_cols, terms), k)


def test_nse_hands_back(RBF, O, gpu):
    """A duplicated point (singular), and Hermite stencils with Dirichlet rows of one entry:
    the rook kernels solve or report what the elimination hands back."""
    from test_oracle import _unit_square_441

    pts = np.random.default_rng(0).random((50, 2))
    pts[1] = pts[0]
    with pinned(RBF, K_NSE):
        with pytest.raises(RBF.SingularException):
            RBF.gradient(pts, k=12)
    pts, isb, nrm, bcs = _unit_square_441()
    adjl = O.knn(pts, pts, 15)
    herm = dict(is_boundary=isb, bc=[RBF.BoundaryCondition(a, b) for a, b in bcs], normals=nrm)
    with pinned(RBF, K_NSE):
        op = RBF.laplacian(pts, basis=RBF.PHS(3, poly_deg=2), adjl=adjl, hermite=herm)
        assert 0 < RBF._lib.last_build_stats()[0] < len(pts) and RBF._lib.last_build_buckets()[1][0] == K_NSE
    ptr, col, wr, _, rc = O.build(pts, pts, adjl, O.basis_struct(3, 2), _op(O, 1, [(0, O.abi.OP_LAP, 0, 0, 1.0)]),
                                  scaled=True, long_double=True, hermite=(isb, bcs[:, 0], bcs[:, 1], nrm))
    assert rc == 0 and np.array_equal(op.row_ptr.cpu().numpy(), ptr) and np.array_equal(op.col.cpu().numpy(), col)
    w = op.vals.cpu().numpy()[0]
    scale = np.maximum.reduceat(np.abs(wr[0]), ptr[:-1])
    err = np.maximum.reduceat(np.abs(w - wr[0]), ptr[:-1])
    assert np.all(err <= 1e-10 * scale), (err / scale).max()


def test_nse_repeated_builds_bit_identical(RBF, gpu):
    """Repeated builds of one operator give the same bits, and so does a captured replay."""
    import torch

    pts = torch.as_tensor(np.random.default_rng(5).random((9001, 3)), device=gpu)
    f = torch.sin(3 * pts[:, 0])
    with pinned(RBF, K_NSE):
        op = RBF.gradient(pts, basis=RBF.PHS(3, poly_deg=2), k=25)
        first = op.vals.clone()
        for _ in range(8):
            op.update_weights()
            assert torch.equal(op.vals, first)
        g = op.capture(f)
        for _ in range(4):
            op.vals.zero_()
            y = g.replay().clone()
            torch.cuda.synchronize()
            assert torch.equal(op.vals, first)
        assert torch.equal(y, g.replay())


@pytest.mark.parametrize("kind,dim,degs,cols,kmax", [(3, 2, (1, 3), "lap", 40), (3, 2, (2, 2), "hess", 36),
                                                    (5, 2, (2, 3), "grad", 40), (3, 3, (2, 2), "gradlap", 40),
                                                    (5, 3, (3, 3), "lap", 50)])
def test_nse_classes_of_uneven_builds(RBF, O, gpu, kind, dim, degs, cols, kmax):
    """Ragged stencils of mixed degree: those within a class run on the elimination kernel
    (null points from 1 to 31, a wavefront's four stencils of different k), the others on the
    rook kernels; every stencil against the extended-precision oracle at max(1e-10, kappa u),
    and a captured replay gives the eager build's bits."""
    import torch

    rng = np.random.default_rng(kind + dim + kmax)
    n = 1501
    pts = rng.random((n, dim))
    L, n_cols, terms = _operator(RBF, O, dim, cols)
    full = O.knn(pts, pts, kmax)
    deg = rng.integers(degs[0], degs[1] + 1, n).astype(np.int8)
    mono = np.array([comb(dim + d, dim) for d in deg])
    ks = np.maximum(rng.integers(mono + 1, kmax + 1), 2)
    edges = [1, 12, 13, 14, 15, 16, 20, 21, 26, 27, 29, 30, 31, 32, 33]
    for i in range(300):  # the edges of the classes, each several times
        ks[i] = min(kmax, mono[i] + edges[i % len(edges)])
    adjl = [full[i, :ks[i]] for i in range(n)]
    op = RBF.RadialBasisOperator(L, pts, basis=RBF.PHS(kind, poly_deg=int(degs[1])), adjl=adjl, poly_deg_map=deg)
    nb, kern = RBF._lib.last_build_buckets()
    nn = ks + mono
    assert nb == [int((nn <= 32).sum()), int(((nn > 32) & (nn <= 64)).sum()), int((nn > 64).sum())]
    w = op.vals.cpu().numpy()
    ptr = op.row_ptr.cpu().numpy()
    u = 2.0 ** -53
    for d in range(degs[0], degs[1] + 1):
        sel = np.flatnonzero(deg == d)
        if not len(sel):
            continue
        aptr = np.concatenate([[0], np.cumsum(ks[sel])])
        adj = (aptr, np.concatenate([adjl[i] for i in sel]))
        b, o = O.basis_struct(kind, d), _op(O, n_cols, terms)
        _, _, wr, _, rc = O.build(pts, pts[sel], adj, b, o, scaled=True, long_double=True)
        assert rc == 0
        kap = O.condition_numbers(pts, pts[sel], adj, b, o)
        for j, i in enumerate(sel):
            g, r = w[:, ptr[i]:ptr[i + 1]], wr[:, aptr[j]:aptr[j + 1]]
            err = (np.abs(g - r).max(1) / np.abs(r).max(1)).max()
            assert err <= max(1e-10, kap[j] * u), (d, ks[i], err, kap[j] * u)
    f = torch.as_tensor(np.sin(3 * pts[:, 0]), device=gpu)
    eager = op.vals.clone()
    g = op.capture(f)
    for _ in range(3):
        op.vals.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(op.vals, eager)


@pytest.mark.parametrize("where", ["front", "back", "apart"])
@pytest.mark.parametrize("kind,dim,deg,nn,cols", [(3, 2, 1, 1, "grad"), (3, 2, 2, 1, "lap"), (3, 2, 2, 2, "lap"),
                                                 (3, 2, 2, 3, "lap"), (3, 2, 2, 6, "hess"), (5, 2, 3, 1, "lap"),
                                                 (5, 2, 3, 2, "grad"), (7, 2, 4, 1, "lap"), (3, 3, 2, 1, "lap"),
                                                 (3, 3, 2, 2, "grad"), (5, 3, 3, 1, "lap"), (5, 3, 3, 2, "gradlap")])
def test_nse_never_accepts_a_repeated_point(RBF, O, gpu, kind, dim, deg, nn, cols, where):
    """Stencils of m + nn points, two of them the same point: singular systems, of which
    rounding leaves pivots of either sign. Every one goes back to the rook kernel, which solves
    or reports it, wherever the pair stands in the stencil and however few points there are."""
    k = comb(dim + deg, dim) + nn
    n = 901
    pts = np.random.default_rng(13 * kind + deg + nn).random((n, dim))
    near = O.knn(pts, pts, k - 1)
    q = {"front": 0, "back": k - 2, "apart": (k - 1) // 2}[where]
    twin = near[:, q:q + 1] + n
    adj = np.concatenate([near[:, :1], twin, near[:, 1:]] if where == "front" else [near, twin], axis=1)
    L, n_cols, terms = _operator(RBF, O, dim, cols)
    with pinned(RBF, K_NSE):
        try:
            RBF.RadialBasisOperator(L, np.concatenate([pts, pts]), eval_points=pts, basis=RBF.PHS(kind, poly_deg=deg),
                                    adjl=list(adj))
        except RBF.SingularException:
            pass
    assert K_NSE in RBF._lib.last_build_buckets()[1]
    assert RBF._lib.last_build_stats()[0] == n
