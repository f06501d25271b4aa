"""Accuracy of the null-space elimination (kernel id 8) beside the kernels it replaced, against
weights assembled and solved in extended precision from the stored coordinates: roundings of
the offsets and of phi, whichever kernel makes them, count as its error."""
import itertools
from math import comb

import numpy as np
import pytest

from test_gpu_nse import K_NSE

pytestmark = pytest.mark.gpu
N = 300


def _stencils(O, dim, k, seed):
    """(cloud, evaluation points, adjacency, offsets): N points of a jittered grid with its faces
    and corners, their nearest neighbours, and the offsets scaled by a power of two to a radius
    of 0.5 to 1."""
    rng = np.random.default_rng(seed)
    m = 30 if dim == 2 else 10
    g = np.stack(np.meshgrid(*[np.linspace(0.0, 1.0, m)] * dim, indexing="ij"), -1).reshape(-1, dim)
    pts = g + rng.uniform(-0.3, 0.3, g.shape) / (m - 1)
    ev = pts[rng.choice(len(pts), N, replace=False)]
    adj = O.knn(pts, ev, k)
    x = pts[adj] - ev[:, None]
    s = np.frexp(np.sqrt((x * x).sum(-1)).max())[1]
    return pts, ev, adj, np.ldexp(x, -s), s


def _monomials(dim, deg):
    return [e for t in range(deg + 1) for e in itertools.product(range(t + 1), repeat=dim) if sum(e) == t]


def _block(x, mono):
    return np.stack([np.prod([x[..., c] ** e for c, e in enumerate(es)], axis=0) for es in mono], -1)


def _columns(dim, cols):
    unit = [tuple(int(i == j) for i in range(dim)) for j in range(dim)]
    return {"lap": ["lap"], "dx": unit[:1], "grad": unit, "gradlap": unit + ["lap"]}[cols]


def _exact(x, p, deg, cols):
    """(columns, N, k) weights and (columns, m) polynomial right-hand sides, extended precision."""
    x = x.astype(np.longdouble)
    n, k, dim = x.shape
    mono = _monomials(dim, deg)
    m = len(mono)
    q = ((x[:, :, None] - x[:, None]) ** 2).sum(-1)
    A = np.zeros((n, k + m, k + m), dtype=np.longdouble)
    A[:, :k, :k] = q ** (p // 2) * np.sqrt(q)
    A[:, :k, k:] = _block(x, mono)
    A[:, k:, :k] = np.swapaxes(A[:, :k, k:], 1, 2)
    r = np.sqrt((x * x).sum(-1))
    terms = _columns(dim, cols)
    B = np.zeros((n, k + m, len(terms)), dtype=np.longdouble)
    for c, t in enumerate(terms):
        if t == "lap":
            B[:, :k, c] = p * (p + 1) * r ** (p - 2)
            B[:, k:, c] = [2.0 * (sorted(e) == [0] * (dim - 1) + [2]) for e in mono]
        else:
            B[:, :k, c] = -p * x[..., t.index(1)] * r ** (p - 2)
            B[:, k:, c] = [float(e == t) for e in mono]
    g = B[0, k:].T.copy()
    at = np.arange(n)
    for j in range(k + m):  # Gaussian elimination with partial pivoting, all stencils at once
        piv = j + np.argmax(np.abs(A[:, j:, j]).astype(float), 1)
        A[at, j], A[at, piv] = A[at, piv].copy(), A[at, j].copy()
        B[at, j], B[at, piv] = B[at, piv].copy(), B[at, j].copy()
        f = A[:, j + 1:, j] / A[:, j, j][:, None]
        A[:, j + 1:, j:] -= f[..., None] * A[:, j, None, j:]
        B[:, j + 1:] -= f[..., None] * B[:, j, None]
    for j in range(k + m - 1, -1, -1):
        B[:, j] -= (A[:, j, j + 1:, None] * B[:, j + 1:]).sum(1)
        B[:, j] /= A[:, j, j][:, None]
    return np.moveaxis(B[:, :k], -1, 0), g


def _operator(RBF, dim, cols):
    return {"lap": RBF.Laplacian, "dx": lambda: RBF.Partial(1, 1), "grad": lambda: RBF.Jacobian(dim),
            "gradlap": lambda: RBF.Stacked(RBF.Jacobian(dim), RBF.Laplacian())}[cols]()


def _weights(RBF, pts, ev, adj, kind, deg, L, kernel):
    rows = adj.shape[1] + comb(pts.shape[1] + deg, pts.shape[1])
    bucket = 0 if rows <= 32 else (1 if rows <= 64 else 2)
    RBF._lib.tune_bucket(bucket, kernel)
    try:
        op = RBF.RadialBasisOperator(L, pts, eval_points=ev, basis=RBF.PHS(kind, poly_deg=deg), adjl=list(adj))
    finally:
        RBF._lib.tune_bucket(bucket, -1)
    assert kernel in RBF._lib.last_build_buckets()[1] and RBF._lib.last_build_stats()[0] == 0
    return op.vals.cpu().numpy().reshape((-1,) + adj.shape)


# kernels: 5, 6 null-space Cholesky, 0, 7 rook; those that took these builds before kernel 8
HIGH = [(3, 2, 3, 20, "lap", 5), (3, 2, 3, 20, "grad", 0), (3, 2, 3, 27, "lap", 5), (3, 2, 3, 30, "grad", 7),
        (5, 2, 3, 20, "dx", 5), (5, 2, 3, 25, "grad", 7), (7, 2, 3, 20, "lap", 5), (7, 2, 4, 30, "grad", 7),
        (3, 3, 2, 27, "lap", 7), (3, 3, 2, 35, "grad", 7), (5, 3, 3, 40, "grad", 7), (5, 3, 3, 40, "lap", 7),
        (5, 3, 3, 45, "gradlap", 7), (7, 3, 3, 40, "lap", 7)]


def test_weights_as_exact_as_the_replaced_kernels(RBF, O, gpu):
    """2-norm of the weights' errors over the stencils of a shape, kernel 8 over the replaced
    kernel, for 10 monomials and more: at most 1 in the geometric mean over the shapes."""
    ratios = []
    for kind, dim, deg, k, cols, other in HIGH:
        pts, ev, adj, x, s = _stencils(O, dim, k, 100 * kind + k + len(cols))
        ref, _ = _exact(x, kind, deg, cols)
        for c, t in enumerate(_columns(dim, cols)):
            ref[c] = np.ldexp(ref[c], -s * (2 if t == "lap" else 1))
        e8, eo = (np.linalg.norm((_weights(RBF, pts, ev, adj, kind, deg, _operator(RBF, dim, cols), kern) - ref).astype(float))
                  for kern in (K_NSE, other))
        print((kind, dim, deg, k, cols), "%.3f" % (e8 / eo))
        ratios.append(e8 / eo)
    assert np.exp(np.mean(np.log(ratios))) <= 1.0, ratios


ALL = [(3, 2, 1, 12, "lap", 6), (3, 2, 2, 7, "lap", 6), (3, 2, 2, 12, "grad", 0), (3, 2, 2, 20, "lap", 6),
       (3, 2, 2, 25, "lap", 5), (3, 2, 2, 32, "dx", 5), (5, 2, 2, 20, "lap", 6), (3, 3, 1, 12, "lap", 6),
       (3, 3, 2, 20, "grad", 7)] + HIGH


def test_polynomial_conditions_as_exact_as_the_replaced_kernels(RBF, O, gpu):
    """Residual of P^T w = L P relative to the stencil's largest weight (what an applied operator
    shows on a smooth field), root mean square over the stencils of a shape, kernel 8 over
    the replaced kernel: at most 1 in the geometric mean over the shapes."""
    ratios = []
    for kind, dim, deg, k, cols, other in ALL:
        pts, ev, adj, x, s = _stencils(O, dim, k, 7 * kind + k + len(cols))
        P = _block(x.astype(np.longdouble), _monomials(dim, deg))
        res = []
        for kern in (K_NSE, other):
            w = _weights(RBF, pts, ev, adj, kind, deg, _operator(RBF, dim, cols), kern).astype(np.longdouble)
            r = []
            for c, t in enumerate(_columns(dim, cols)):
                wc = np.ldexp(w[c], s * (2 if t == "lap" else 1))
                g = [2.0 * (sorted(e) == [0] * (dim - 1) + [2]) if t == "lap" else float(e == t) for e in _monomials(dim, deg)]
                r.append(((P * wc[:, :, None]).sum(1) - g) / np.abs(wc).max(1)[:, None])
            res.append(float(np.sqrt((np.array(r) ** 2).mean())))
        print((kind, dim, deg, k, cols), "%.3f" % (res[0] / res[1]))
        ratios.append(res[0] / res[1])
    assert np.exp(np.mean(np.log(ratios))) <= 1.0, ratios
