"""Workloads that a user of the framework runs, for timing its public entry points.

`listed()` names twelve of them, `draw(rng)` gives more of the same ranges. A case's
"kind" says which calls a pass makes:

  construct  an operator from points (k-NN and weight build), then one apply
  update     weights rebuilt for a kept operator (`update_weights`): points that moved,
             or the build stage of a program that keeps its neighbour lists
  apply      a kept operator on fields
  replay     build and apply recorded once (`capture`) and replayed each time step
  train      forward and backward pass of the weight surrogate on one batch

Point clouds are quasi-uniform, as node generators make them for RBF-FD: jittered grids,
a jittered grid mapped conformally onto an annular sector (density x10 across it),
Halton points, and a graded sunflower disk with boundary nodes on its circle; the regrid
takes its sources uniformly random.
"""
import itertools
import math
import pathlib

import numpy as np
import torch

import rbfx_loader

R = rbfx_loader.load()
DEV = "cuda:0"
MODEL = pathlib.Path(R.__file__).resolve().parent / "models" / "surrogate_lap2d_phs3_k20.npz"


def _case(name, kind, op, cloud, dim, n, basis, deg, k, **more):
    c = {"name": name, "kind": kind, "op": op, "cloud": cloud, "dim": dim, "n": n, "basis": basis, "deg": deg,
         "k": k, "fields": 0, "dtype": "float64", "precision": "fp64"}
    c.update(more)
    return c


def listed():
    return [
        # the smallest full call: a 30 x 30 cloud with the default basis and stencil
        # size, where launches, synchronisations and host work are all there is
        _case("construct_lap2d_900", "construct", "laplacian", "jitter", 2, 900, "phs3", 2, 12),
        # one right-hand side evaluation of a small model: a single kept apply
        _case("apply_lap2d_4900", "apply", "laplacian", "jitter", 2, 4900, "phs5", 3, 20),
        # a time step on a small moving cloud: build and apply as one graph replay
        _case("replay_lap2d_10k", "replay", "laplacian", "jitter", 2, 10_000, "phs3", 2, 20, fields=1),
        # an ordinary three-dimensional cloud with the default basis: gradient from
        # scratch and its first evaluation
        _case("construct_grad3d_100k", "construct", "gradient", "halton", 3, 100_000, "phs3", 2, 20, fields=1),
        # single precision in and out, three output columns, a higher order basis
        _case("construct_hess2d_120k_f32", "construct", "hessian", "jitter", 2, 120_001, "phs5", 3, 20, fields=1,
              dtype="float32"),
        # the large two-dimensional weight build
        _case("update_lap2d_4M", "update", "laplacian", "graded", 2, 4_000_000, "phs3", 2, 20),
        # the surrogate with its acceptance test and fallback solve
        _case("update_lap2d_1M_learned", "update", "laplacian", "graded", 2, 1_000_000, "phs3", 2, 20,
              precision="learned"),
        # large three-dimensional systems, several operators on one factorisation
        _case("update_gradlap3d_2M", "update", "gradlap", "jitter", 3, 2_000_376, "phs5", 3, 40),
        # uneven stencils (k from the local density, degree 3 beside the boundary) with
        # Neumann rows on the circle
        _case("update_disk_1M3", "update", "dx_d2y", "disk", 2, 1_290_000, "phs3", 3, 60),
        # interpolation between two large clouds with a nearly flat kernel
        _case("update_regrid3d_8M", "update", "regrid", "random", 3, 4_000_000, "imq", 1, 30, targets=8_000_000),
        # sixteen fields moved between those clouds
        _case("apply_regrid3d_8M_16", "apply", "regrid", "random", 3, 4_000_000, "imq", 1, 30, targets=8_000_000,
              fields=16),
        # forward and backward pass of the surrogate at its training batch
        _case("train_surrogate_4096", "train", "laplacian", "random", 2, 4096, "phs3", 2, 20),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# (dim, basis, degree, stencil sizes): the default size of the pairing and others in use
_PAIRINGS = [(2, "phs3", 2, (12, 13, 20, 25)), (2, "phs3", 3, (20, 27, 30)), (2, "phs5", 3, (20, 25)),
             (2, "phs7", 4, (30,)), (3, "phs3", 2, (20, 27, 35)), (3, "phs5", 3, (40, 45)), (3, "phs3", 1, (10, 15))]


def draw(rng):
    kind = rng.choice(["construct", "construct", "update", "update", "apply", "replay", "disk", "regrid"])
    if kind == "disk":
        return _drawn("update", "dx_d2y", "disk", 2, _log_int(rng, 20_000, 400_000), "phs3", 3, 60)
    if kind == "regrid":
        n = _log_int(rng, 20_000, 1_000_000)
        return _drawn(rng.choice(["update", "apply"]), "regrid", "random", 3, n, "phs3", 2, rng.choice([20, 25, 30]),
                      targets=_log_int(rng, n // 2, 2 * n), fields=rng.choice([1, 3, 8, 16]))
    dim, basis, deg, ks = rng.choice(_PAIRINGS)
    op = rng.choice(["laplacian", "gradient", "partial"] + (["hessian"] if deg >= 2 else []))
    top = {"construct": 300_000, "update": 1_500_000, "apply": 1_000_000, "replay": 60_000}[kind]
    low = {"construct": 225, "update": 20_000, "apply": 1_000, "replay": 1_000}[kind]
    cloud = rng.choice(["jitter", "graded"] if dim == 2 else ["jitter", "halton"])
    fields = 0 if kind == "update" else (1 if op != "laplacian" and op != "partial" else rng.choice([1, 1, 2, 5, 8]))
    return _drawn(kind, op, cloud, dim, max(_log_int(rng, low, top), 3 * max(ks)), basis, deg, rng.choice(ks),
                  fields=fields, dtype="float32" if kind == "construct" and rng.random() < 0.25 else "float64")


def _drawn(*a, **more):
    c = _case("", *a, **more)
    del c["name"]
    return c


# ------------------------------------------------------------------ inputs
def _generator(seed, device=DEV):
    return torch.Generator(device=device).manual_seed(int(seed))


def _jitter(n, dim, g):
    """n points of a jittered grid on the unit square or cube, in a scattered order
    unless the grid holds exactly n."""
    m = round(n ** (1.0 / dim))
    while m ** dim < n:
        m += 1
    lin = torch.linspace(0.0, 1.0, m, dtype=torch.float64, device=DEV)
    p = torch.stack(torch.meshgrid(*[lin] * dim, indexing="ij"), -1).reshape(-1, dim)
    p = p + (0.6 * torch.rand(p.shape, dtype=torch.float64, device=DEV, generator=g) - 0.3) / (m - 1)
    if m ** dim > n:
        p = p[torch.randperm(m ** dim, device=DEV, generator=g)[:n]]
    return p.contiguous()


def _graded(n, g):
    """A jittered grid in (ln r, angle) mapped onto an annular sector: density x10."""
    side = 0.5 * math.log(10.0)
    p = _jitter(n, 2, g) * side
    p = p[torch.randperm(n, device=DEV, generator=g)]
    r = torch.exp(p[:, 0])
    return torch.stack([r * torch.cos(p[:, 1]), r * torch.sin(p[:, 1])], 1).contiguous()


def _halton(n, dim, g):
    i = torch.arange(1, n + 1, dtype=torch.int64, device=DEV)
    cols = []
    for b in (2, 3, 5)[:dim]:
        v, f, j = torch.zeros(n, dtype=torch.float64, device=DEV), 1.0, i.clone()
        while f > 1.0 / (b * n):
            f /= b
            v += f * (j % b)
            j //= b
        cols.append(v)
    shift = torch.rand(dim, dtype=torch.float64, device=DEV, generator=g)
    return ((torch.stack(cols, 1) + shift) % 1.0).contiguous()


def _disk(n, g):
    """(points, number of boundary nodes): a sunflower disk graded towards its centre,
    the last points evenly spaced on the circle; without a generator the plain pattern."""
    gamma = 1.4
    edge = math.sqrt(math.pi * gamma / n)  # spacing at the rim
    nb = int(2 * math.pi / (edge * 1.1))
    i = torch.arange(n - nb, dtype=torch.float64, device=DEV)
    jit = 0.3 * torch.rand(n - nb, dtype=torch.float64, device=DEV, generator=g) if g is not None else 0.15
    s = torch.sqrt((i + 0.5 + jit) / (n - nb + 0.5 * nb))
    r = s ** gamma * (1.0 - 0.7 * edge)
    th = i * (math.pi * (3.0 - math.sqrt(5.0)))
    b = torch.arange(nb, dtype=torch.float64, device=DEV) * (2.0 * math.pi / nb)
    turn = torch.zeros(1, dtype=torch.float64, device=DEV)
    if g is not None:
        turn = 2.0 * math.pi * torch.rand(1, dtype=torch.float64, device=DEV, generator=g)
    inner = torch.stack([r * torch.cos(th + turn), r * torch.sin(th + turn)], 1)
    return torch.cat([inner, torch.stack([torch.cos(b + turn), torch.sin(b + turn)], 1)]).contiguous(), nb


def _points(case, seed):
    g = _generator(seed)
    if case["cloud"] == "graded":
        return _graded(case["n"], g)
    if case["cloud"] == "halton":
        return _halton(case["n"], case["dim"], g)
    if case["cloud"] == "random":
        return torch.rand((case["n"], case["dim"]), dtype=torch.float64, device=DEV, generator=g)
    return _jitter(case["n"], case["dim"], g)


def _dtype(case):
    return torch.float32 if case["dtype"] == "float32" else torch.float64


def _fields(case, points):
    """Smooth fields with a few wavelengths across the cloud, (n,) or (n, fields)."""
    f = max(1, case["fields"])
    w = torch.arange(1, f + 1, dtype=torch.float64, device=DEV)
    v = torch.sin(4.0 * points[:, :1] + 0.3 * w) * torch.cos((3.0 + 0.2 * w) * points[:, 1:2] + points[:, -1:])
    return (v[:, 0] if f == 1 else v).contiguous().to(_dtype(case))


def _basis(case):
    name, deg = case["basis"], case["deg"]
    return R.IMQ(3.0, poly_deg=deg) if name == "imq" else R.PHS(int(name[3:]), poly_deg=deg)


def _operator(case):
    d = case["dim"]
    return {"laplacian": R.Laplacian, "partial": lambda: R.Partial(1, 1), "gradient": lambda: R.Jacobian(d),
            "hessian": lambda: R.Hessian(d), "gradlap": lambda: R.Stacked(R.Jacobian(d), R.Laplacian()),
            "dx_d2y": lambda: R.Partial(1, 1) + R.Partial(2, 2), "regrid": R.Regrid}[case["op"]]()


def _disk_operator(case, seed):
    pts, nb = _disk(case["n"], _generator(seed))
    n = pts.shape[0]
    plain, _ = _disk(case["n"], None)  # the sizes follow the pattern, not its perturbation
    d12 = (plain - plain[R._lib.knn(plain, plain, 13)[:, -1].long()]).norm(dim=1)
    kk = torch.clamp((24 * (d12.median() / d12) ** 2).long(), 12, case["k"])
    kk[n - nb:] = case["k"]
    ptr = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    ptr[1:] = torch.cumsum(kk, 0)
    idx = R._lib.knn(pts, pts, case["k"], q_ptr=ptr)
    hits = torch.zeros(idx.numel() + 1, dtype=torch.int64, device=DEV)
    hits[1:] = torch.cumsum((idx >= n - nb).long(), 0)
    touch = hits[ptr[1:]] > hits[ptr[:-1]]
    isb = np.zeros(n, dtype=bool)
    isb[n - nb:] = True
    herm = R.Hermite(isb, [R.Neumann()] * nb, pts[n - nb:].cpu().numpy())
    return R.RadialBasisOperator(_operator(case), pts, basis=_basis(case), adjl=(ptr, idx), hermite=herm,
                                 poly_deg_map=torch.where(touch, 3, 2).to(torch.int8))


def _kept_operator(case, seed, points):
    if case["cloud"] == "disk":
        return _disk_operator(case, seed)
    kw = {"basis": _basis(case), "k": case["k"]}
    if case["precision"] == "learned":
        kw.update(precision="learned", model=R.LearnedModel.load(MODEL))
    if case["op"] == "regrid":
        m = round(case["targets"] ** (1.0 / case["dim"]))
        while m ** case["dim"] < case["targets"]:
            m += 1
        return R.regrid(points, _jitter(case["targets"], case["dim"], _generator(seed + 7)).clamp(0.0, 1.0), **kw)
    return R.RadialBasisOperator(_operator(case), points, **kw)


def prepare(case, seed):
    if case["kind"] == "train":
        return _prepare_train(case, seed)
    pts = None if case["cloud"] == "disk" else _points(case, seed)
    s = {"case": case}
    if case["kind"] == "construct":
        s["points"] = pts.to(_dtype(case))
        s["f"] = _fields(case, pts) if case["fields"] else None
        return s
    s["op"] = _kept_operator(case, seed, pts)
    if case["kind"] in ("apply", "replay"):
        s["f"] = _fields(case, pts)
    if case["kind"] == "replay":
        s["graph"] = s["op"].capture(s["f"])
    return s


def _prepare_train(case, seed):
    A, L = R._abi, R._lib
    m = R.LearnedModel.load(MODEL)
    X, Y, rw = R.learned.training_set(case["n"], seed=int(seed) % (1 << 31))
    t = ((Y - m.out_mean) / m.out_std).float().contiguous()
    return {"case": case, "m": m, "X": X, "t": t, "rw": rw,
            "ws": torch.empty(L.mlp_workspace_bytes(case["n"]), dtype=torch.uint8, device=DEV),
            "grads": torch.empty(A.MLP_N_PARAMS, dtype=torch.float32, device=DEV),
            "loss": torch.zeros(1, dtype=torch.float32, device=DEV),
            "y": torch.empty((case["n"], A.MLP_OUT_PAD), dtype=torch.float32, device=DEV)}


# ------------------------------------------------------------------ one pass
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "construct":
        op = R.RadialBasisOperator(_operator(case), s["points"], basis=_basis(case), k=case["k"])
        out = {"adj": op.adj_idx}
        if case["dtype"] == "float64":
            out["w"] = op.vals
        if s["f"] is not None:
            out["y"] = op(s["f"])
        return out
    if kind == "update":
        s["op"].update_weights()
        return s["op"].vals
    if kind == "apply":
        return s["op"](s["f"])
    if kind == "replay":
        return {"y": s["graph"].replay(), "w": s["op"].vals}
    m = s["m"]
    R._lib.mlp_run(s["X"], m.params, m.wbf16, s["ws"], case["n"], target=s["t"], grads=s["grads"], loss=s["loss"],
                   y_out=s["y"], n_out=m.n_out, row_weight=s["rw"])
    return {"y": s["y"], "grads": s["grads"], "loss": s["loss"]}


# ------------------------------------------------------------------ least work
def work(case):
    """Bytes: inputs once, outputs once. Flops: the factorisation and the solves of each
    stencil's (k + m)-row symmetric system, two per stored weight of an apply."""
    if case["kind"] == "train":
        macs = 80 * 256 + 2 * 256 * 256 + 256 * 26
        return {"bytes": 4 * 151_000 * 2 + case["n"] * (2 * 128 + 4 * 26 + 4 * 32), "flops": 6.0 * macs * case["n"]}
    d, n, k = case["dim"], case["n"], case["k"]
    ne = case.get("targets", n)
    cols = {"gradient": d, "hessian": d * (d + 1) // 2, "gradlap": d + 1}.get(case["op"], 1)
    if case["cloud"] == "disk":
        k = 24  # the median stencil
    m = math.comb(d + case["deg"], d)
    f = max(1, case["fields"])
    fb = 4 if case["dtype"] == "float32" else 8
    nnz = ne * k
    b = fl = 0.0
    if case["kind"] in ("construct", "update", "replay"):
        b += 8.0 * d * (n + (ne if ne != n or case["op"] == "regrid" else 0)) + 4.0 * nnz + 8.0 * cols * nnz
        fl += ne * ((k + m) ** 3 / 3.0 + 2.0 * (k + m) ** 2 * cols)
    if case["kind"] in ("apply", "replay") or (case["kind"] == "construct" and case["fields"]):
        b += fb * f * (n + cols * ne) + (4.0 + 8.0 * cols) * nnz
        fl += 2.0 * nnz * cols * f
    return {"bytes": b, "flops": fl}


# ------------------------------------------------------------------ 64-bit results
def _exact_knn(x, q, k):
    """Indices of the k nearest points, ascending, lower index first on ties."""
    out = np.empty((len(q), k), dtype=np.int64)
    xd, step = x.to(DEV), max(64, int(2.5e7 // len(x)))
    for s in range(0, len(q), step):
        d2 = torch.zeros((min(step, len(q) - s), len(x)), dtype=torch.float64, device=DEV)
        for c in range(x.shape[1]):
            d2 += (xd[None, :, c] - q[s:s + step, c].to(DEV)[:, None]) ** 2
        v, i = torch.topk(d2, k, largest=False)
        i = i.gather(1, torch.argsort(i, 1))
        v = d2.gather(1, i)
        out[s:s + step] = i.gather(1, torch.sort(v, dim=1, stable=True)[1]).cpu().numpy()
    return out


def _monomials(dim, deg):
    return [e for t in range(deg + 1) for e in itertools.product(range(t + 1), repeat=dim) if sum(e) == t]


def _columns(case):
    """Per operator column its terms (derivative orders per dimension, or "lap")."""
    d = case["dim"]
    unit = [tuple(int(i == j) for i in range(d)) for j in range(d)]
    return {"laplacian": [["lap"]], "partial": [[unit[0]]], "gradient": [[u] for u in unit],
            "gradlap": [[u] for u in unit] + [["lap"]], "regrid": [[(0,) * d]],
            "hessian": [[tuple(a + b for a, b in zip(unit[i], unit[j]))] for i in range(d) for j in range(i, d)],
            }[case["op"]]


def _phi_term(p, D, term, dim):
    """The term applied to r^p at offsets D (..., dim) of the centre; the Laplacian of a
    spline takes p (p + 1) r^(p - 2) in every dimension, as the reference defines it."""
    r = np.sqrt((D * D).sum(-1))
    if term == "lap":
        return p * (p + 1) * r ** (p - 2)
    if sum(term) == 0:
        return r ** p
    if sum(term) == 1:
        return p * D[..., term.index(1)] * r ** (p - 2)
    low = 1.0 / np.where(r > 0, r, 1.0) if p == 3 else r ** (p - 4)
    ij = [i for i, t in enumerate(term) for _ in range(t)]
    v = p * (p - 2) * D[..., ij[0]] * D[..., ij[1]] * low
    return v + p * r ** (p - 2) if ij[0] == ij[1] else v


def _poly_term(e, term, dim):
    """The term applied to the monomial x^e at the origin."""
    if term == "lap":
        return sum(2.0 for i in range(dim) if e == tuple(2 * int(i == j) for j in range(dim)))
    return float(math.prod(math.factorial(t) for t in term)) if e == term else 0.0


def _exact_weights(case, x, ev, adj):
    """(columns, stencils, k) in extended precision where numpy has it: each scaled
    system solved in 64 bits and corrected once from an extended residual."""
    dim, k, p, mono = case["dim"], case["k"], int(case["basis"][3:]), _monomials(case["dim"], case["deg"])
    cols, m = _columns(case), len(_monomials(case["dim"], case["deg"]))
    W = np.empty((len(cols), len(ev), k), dtype=np.longdouble)
    step = 4096
    for s in range(0, len(ev), step):
        D = (x[adj[s:s + step]] - ev[s:s + step, None]).astype(np.longdouble)
        h = np.sqrt((D * D).sum(-1).max(1))
        D = D / h[:, None, None]
        A = np.zeros((len(D), k + m, k + m), dtype=np.longdouble)
        q = np.zeros((len(D), k, k), dtype=np.longdouble)
        for c in range(dim):
            q += (D[:, :, None, c] - D[:, None, :, c]) ** 2
        A[:, :k, :k] = q ** (p // 2) * np.sqrt(q)
        B = np.zeros((len(D), k + m, len(cols)), dtype=np.longdouble)
        for a, e in enumerate(mono):
            v = np.ones(D.shape[:2], dtype=np.longdouble)
            for c in range(dim):
                v = v * D[..., c] ** e[c]
            A[:, :k, k + a] = v
            A[:, k + a, :k] = v
            for j, terms in enumerate(cols):
                B[:, k + a, j] = sum(_poly_term(e, t, dim) for t in terms)
        for j, terms in enumerate(cols):
            B[:, :k, j] = sum(_phi_term(p, -D, t, dim) for t in terms)
        A64 = A.astype(np.float64)
        X = np.linalg.solve(A64, B.astype(np.float64)).astype(np.longdouble)
        res = np.stack([B[..., j] - (A * X[:, None, :, j]).sum(-1) for j in range(len(cols))], -1)
        X = X + np.linalg.solve(A64, res.astype(np.float64))
        for j, terms in enumerate(cols):
            o = 2 if terms[0] == "lap" else sum(terms[0])
            W[j, s:s + step] = X[:, :k, j] / h[:, None] ** o
    return W


def exact(case, seed):
    if case["kind"] == "train":
        return _exact_train(case, seed)
    cols = 0 if case["cloud"] == "disk" else len(_columns(case))
    ne = case.get("targets", case["n"])
    cost = ne * (case["k"] + 15) ** 2 * (1 + 0.3 * cols)  # about: a second for every 3e7
    if case["cloud"] == "disk" or case["basis"] == "imq" or case["precision"] == "learned" or cost > 3.5e8 \
            or ne * case["n"] > 2e10:
        return None
    pts = _points(case, seed)
    f = _fields(case, pts).double().cpu().numpy()
    if case["kind"] == "construct":
        pts = pts.to(_dtype(case)).double()
    ev = pts
    if case["op"] == "regrid":
        ev = _jitter(ne, case["dim"], _generator(seed + 7)).clamp(0.0, 1.0)
    adj = _exact_knn(pts, ev, case["k"])
    W = _exact_weights(case, pts.cpu().numpy(), ev.cpu().numpy(), adj)
    w = W.reshape(len(W), -1).astype(np.float64)
    if case["kind"] == "update":
        return w
    F = (f[:, None] if f.ndim == 1 else f).astype(np.longdouble)
    Y = np.stack([np.stack([(Wc * F[adj, j]).sum(-1) for j in range(F.shape[1])], -1) for Wc in W])
    Y = Y.astype(np.float64)  # (columns, stencils, fields)
    if case["kind"] == "replay":
        return {"y": Y, "w": w}
    y = Y[..., 0] if f.ndim == 1 else Y
    if case["op"] in ("laplacian", "partial", "regrid"):
        y = y[0]
    elif case["op"] == "gradient":
        y = np.moveaxis(y, 0, -1)
    else:
        d, full = case["dim"], None
        full = np.empty(y.shape[1:] + (d, d))
        for c, (i, j) in enumerate((i, j) for i in range(d) for j in range(i, d)):
            full[..., i, j] = full[..., j, i] = y[c]
        y = full
    if case["kind"] == "apply":
        return y
    out = {"adj": adj.astype(np.int32)}
    if case["dtype"] == "float64":
        out["w"] = w
    if case["fields"]:
        out["y"] = y
    return out


def _exact_train(case, seed):
    """The network and its gradients in 64 bits without rounding in between."""
    A = R._abi
    s = _prepare_train(case, seed)
    m, n = s["m"], case["n"]
    par = s["m"].params.double().cpu().requires_grad_(True)
    h = s["X"].double().cpu()
    for l in range(A.MLP_LAYERS):
        K, N, o = A.mlp_k(l), A.mlp_n(l), A.mlp_w_off(l)
        h = h @ par[o:o + N * K].reshape(N, K).T + par[o + N * K:o + N * K + N]
        if l < A.MLP_LAYERS - 1:
            h = torch.nn.functional.gelu(h, approximate="tanh")
    d = h[:, :m.n_out] - s["t"].double().cpu()
    loss = ((d * d).sum(1) * s["rw"].double().cpu()).sum() / (n * m.n_out)
    loss.backward()
    return {"y": h.detach(), "grads": par.grad, "loss": loss.detach().reshape(1)}
