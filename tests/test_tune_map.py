"""Builds that keep out the null-space elimination (kernel 8), because the caller wants the
multipliers, beside plain builds of the same shape: neither decides the other's kernel, in
memory or through a saved map. Maps written before such entries existed still load."""
import ctypes as C
import pathlib

import numpy as np
import pytest

K_NSE = 8


def test_map_lines_without_gpu(RBF, tmp_path):
    """A map line has ten fields, and an eleventh, 1, for a build without kernel 8."""
    lib = C.CDLL(str(pathlib.Path(RBF.__file__).parent / "librbfx.so"))
    lib.rbfx_tune_load.argtypes = [C.c_char_p]
    lib.rbfx_tune_save.argtypes = [C.c_char_p]
    lib.rbfx_tune_reset()
    f = tmp_path / "map.txt"
    f.write_text("# kernels\n2 1 0 0 20 6 3 0 1 8\n2 1 0 0 20 6 3 0 1 6 1\n2 1 0 3 60 10 3 0 0 2 1\n2 1 0 1 30 6 3 0 1 5 # k\n")
    assert lib.rbfx_tune_load(str(f).encode()) == 0
    assert lib.rbfx_tune_save(str(f).encode()) == 0
    lines = sorted(l for l in f.read_text().splitlines() if not l.startswith("#"))
    assert lines == sorted(["2 1 0 0 20 6 3 0 1 8", "2 1 0 0 20 6 3 0 1 6 1", "2 1 0 3 60 10 3 0 0 2 1", "2 1 0 1 30 6 3 0 1 5"])
    for line in ("2 1 0 0 20 6 3 0 1\n", "2 1 0 0 20 6 3 0 1 9 1\n", "2 1 0 3 60 10 3 0 0 5 1\n"):
        f.write_text(line)
        assert lib.rbfx_tune_load(str(f).encode()) != 0
    assert lib.rbfx_tune_reset() == 0


def _build(RBF, gpu, pts, idx, kmax, multipliers, ptr=None):
    """One FP64 Laplacian build through the C ABI, with or without multipliers."""
    import torch

    A = RBF._abi
    n = pts.shape[0]
    nnz = idx.numel()
    vals = torch.empty(nnz, dtype=torch.float64, device=gpu)
    lam = torch.empty(n * 6, dtype=torch.float64, device=gpu) if multipliers else None
    a = A.BuildArgs()
    a.dim, a.k, a.n_data, a.n_eval = 2, kmax, n, n
    a.data = a.eval = pts.data_ptr()
    a.adj_idx = idx.data_ptr()
    a.adj_ptr = a.out_ptr = None if ptr is None else ptr.data_ptr()
    a.basis = A.Basis(3, 2, 0.0)
    a.op = A.make_operator(1, [(0, A.OP_LAP, 0, 0, 1.0)])
    a.out_val, a.out_nnz = vals.data_ptr(), nnz
    a.out_lambda = None if lam is None else lam.data_ptr()
    a.stream = RBF._lib.stream_ptr(gpu).value
    rc, _ = RBF._lib.build_weights(a, gpu)
    assert rc == 0, RBF._lib.last_error()
    return vals


@pytest.mark.gpu
@pytest.mark.parametrize("multipliers_first", [True, False])
def test_uniform_builds_with_and_without_multipliers(RBF, gpu, tmp_path, multipliers_first):
    import torch

    pts = torch.as_tensor(np.random.default_rng(1).random((6000, 2)), device=gpu)
    idx = RBF._lib.knn(pts, pts, 20)
    path = tmp_path / "map.txt"
    RBF._lib.tune_reset()
    try:
        kern, tuned = {}, {}
        for rnd in range(3):
            for m in ((True, False) if multipliers_first else (False, True)):
                _build(RBF, gpu, pts, idx, 20, m)
                kern[m], tuned[m] = RBF._lib.last_build_buckets()[1][0], RBF._lib.last_build_stats()[1]
                if rnd:
                    assert tuned[m] == 0  # (timed once each, then kept; also through a saved map)
            assert kern[False] == K_NSE and kern[True] in (0, 5, 6, 7), kern
            if rnd == 1:
                RBF._lib.tune_save(path)
                RBF._lib.tune_reset()
                RBF._lib.tune_load(path)
        rows = [l.split() for l in path.read_text().splitlines() if not l.startswith("#")]
        assert sorted(len(r) for r in rows) == [10, 11]
        assert [r[9] for r in rows if len(r) == 10] == [str(K_NSE)]
    finally:
        RBF._lib.tune_reset()


@pytest.mark.gpu
def test_uneven_builds_with_and_without_multipliers(RBF, gpu, tmp_path):
    """Launch plans are entries of their own too: one launch kept for builds with multipliers
    leaves the plain builds their null-space classes; a line without the eleventh field
    serves both, as it did."""
    import torch

    rng = np.random.default_rng(2)
    n = 3000  # (too few to be timed)
    pts = torch.as_tensor(rng.random((n, 2)), device=gpu)
    ptr = torch.zeros(n + 1, dtype=torch.int64, device=gpu)
    ptr[1:] = torch.cumsum(torch.as_tensor(rng.integers(12, 41, n), device=gpu), 0)
    idx = RBF._lib.knn(pts, pts, 40, q_ptr=ptr)
    path = tmp_path / "map.txt"
    line = "2 1 0 3 40 6 3 0 0 2"  # dim n_cols precision bucket kmax m basis hermite uniform plan
    try:
        for text, plans in (("", {True: 1, False: 1}), (line + " 1", {True: 2, False: 1}), (line, {True: 2, False: 2})):
            RBF._lib.tune_reset()
            path.write_text(text + "\n")
            RBF._lib.tune_load(path)
            for m in (True, False):
                _build(RBF, gpu, pts, idx, 40, m, ptr)
                st = RBF._lib.last_build_stats()
                assert st[2] == plans[m] and (st[3] > n // 2) == (not m and plans[m] == 1), (text, m, st)
    finally:
        RBF._lib.tune_reset()


@pytest.mark.gpu
def test_small_builds_of_several_columns_stay_on_the_rook_kernel(RBF, gpu):
    """Up to 32 rows and fewer stencils than are timed: the same kernel and bits whether or not a
    larger build of the shape has put kernel 8 into the map; a captured step too."""
    import torch

    pts = torch.as_tensor(np.random.default_rng(3).random((6000, 2)), device=gpu)
    small = pts[:1500].contiguous()
    RBF._lib.tune_reset()
    try:
        first = RBF.gradient(small, k=20)
        assert RBF._lib.last_build_buckets()[1][0] == 0
        RBF.gradient(pts, k=20)
        assert RBF._lib.last_build_buckets()[1][0] == K_NSE
        again = RBF.gradient(small, k=20)
        assert RBF._lib.last_build_buckets()[1][0] == 0
        assert torch.equal(first.vals, again.vals)
        g = again.capture(torch.sin(small[:, 0]))
        for _ in range(3):
            again.vals.zero_()
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(again.vals, first.vals)
    finally:
        RBF._lib.tune_reset()
