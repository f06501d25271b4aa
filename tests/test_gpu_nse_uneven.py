"""Uneven builds beside the null-space classes: the classes solve the stencils that belong to
them."""
from math import comb

import numpy as np
import pytest

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
