"""Uneven builds beside the null-space classes: the classes solve the stencils that belong to
them, and a build that times its kernels (on what the classes leave, or on everything where
that is little) gives weights within the same bound as the build that uses its choice."""
from math import comb

import numpy as np
import pytest

from test_gpu_build import _op

pytestmark = pytest.mark.gpu


def _ragged(O, dim, degs, kmax, n, seed, reach=1):
    rng = np.random.default_rng(seed)
    pts = rng.random((n, dim))
    full = O.knn(pts, pts, kmax)
    deg = rng.integers(degs[0], degs[1] + 1, n).astype(np.int8)
    mono = np.array([comb(dim + d, dim) for d in deg])
    ks = rng.integers(mono + reach, kmax + 1)
    return pts, [full[i, :ks[i]] for i in range(n)], deg, mono, ks


@pytest.mark.parametrize("kind,dim,degs,which,cols,kmax,last", [
    (3, 2, (1, 3), "laplacian", 1, 45, {6: 31, 10: 31}), (5, 2, (2, 3), "jacobian", 2, 45, {10: 30}),
    (3, 3, (2, 2), "jacobian", 3, 40, {10: 26}), (5, 3, (3, 3), "laplacian", 1, 50, {20: 26})])
def test_classes_solve_the_stencils_that_belong_to_them(RBF, O, gpu, kind, dim, degs, which, cols, kmax, last):
    pts, adjl, deg, mono, ks = _ragged(O, dim, degs, kmax, 2003, kind + dim)
    L = RBF.Laplacian() if which == "laplacian" else RBF.Jacobian(dim)
    RBF._lib.tune_reset()
    RBF.RadialBasisOperator(L, pts, basis=RBF.PHS(kind, poly_deg=degs[1]), adjl=adjl, poly_deg_map=deg)
    own = sum(int(((mono == m) & (ks - m <= top)).sum()) for m, top in last.items())
    back, _, plan, solved = RBF._lib.last_build_stats()[:4]
    assert plan == 1 and own > 500 and back <= own // 20
    assert solved == own - back


@pytest.mark.parametrize("share", [0.5, 0.95])
def test_first_build_and_the_tuned_one_after_it(RBF, O, gpu, share):
    """60,000 stencils of degree 2 or 3 with 12 to 64 points, more than 4,096 of every size (0.95:
    the classes leave fewer of the small ones). 60 stencils of each size against the
    extended-precision oracle at max(1e-10, kappa u)."""
    import torch

    rng = np.random.default_rng(23)
    n = 60_000
    pts = rng.random((n, 2))
    x = torch.as_tensor(pts, device=gpu)
    full = RBF._lib.knn(x, x, 64).cpu().numpy()
    deg = rng.integers(2, 4, n).astype(np.int8)
    mono = np.where(deg == 2, 6, 10)
    ks = np.where(rng.random(n) < share, rng.integers(12, 33, n), rng.integers(42, 65, n))
    ks[:9000] = rng.integers(56, 65, 9000)
    adjl = [full[i, :ks[i]] for i in range(n)]
    nn = ks + mono
    sizes = [nn <= 32, (nn > 32) & (nn <= 64), nn > 64]
    assert min(int(s.sum()) for s in sizes) > 4096

    def build():
        return RBF.laplacian(pts, basis=RBF.PHS(3, poly_deg=3), adjl=adjl, poly_deg_map=deg, device=gpu)

    RBF._lib.tune_reset()
    first = build()
    timed, plan = RBF._lib.last_build_stats()[1:3]
    assert timed > 0
    second = build()
    assert RBF._lib.last_build_stats()[1] == 0 and RBF._lib.last_build_stats()[2] == plan
    ptr = first.row_ptr.cpu().numpy()
    got = [op.vals.cpu().numpy()[0] for op in (first, second)]
    u = 2.0 ** -53
    for s in sizes:
        for d in (2, 3):
            sel = np.flatnonzero(s & (deg == d))[:30]
            aptr = np.concatenate([[0], np.cumsum(ks[sel])])
            adj = (aptr, np.concatenate([adjl[i] for i in sel]))
            b, o = O.basis_struct(3, d), _op(O, 1, [(0, O.abi.OP_LAP, 0, 0, 1.0)])
            _, _, wr, _, rc = O.build(pts, pts[sel], adj, b, o, scaled=True, long_double=True)
            assert rc == 0
            kap = O.condition_numbers(pts, pts[sel], adj, b, o)
            for j, i in enumerate(sel):
                r = wr[0, aptr[j]:aptr[j + 1]]
                for w in got:
                    err = np.abs(w[ptr[i]:ptr[i + 1]] - r).max() / np.abs(r).max()
                    assert err <= max(1e-10, kap[j] * u), (d, ks[i], err, kap[j] * u)
