"""Performance cases of npbcg: what a program has the library do, at the sizes it is used at.

Every case goes through the public Python front end of the C ABI.  A case is a dict with a
``kind``:

* ``power``      the NPB benchmark's timed loop (``Context.power``) from x = 1, for the orders of
                 the NPB classes and between them;
* ``conj_grad``  one drop-in ``conj_grad`` on host arrays, matrix check included;
* ``solve``      a kept context solving for several right-hand sides in turn, to 1e-10;
* ``oneoff``     a host CSR to its solution and nothing kept: create, solve, destroy;
* ``learned``    a kept context: network inference for its matrix, then solves with the
                 learned preconditioner;
* ``train_grad`` loss, parameter gradient and (g, h) of one training system;
* ``batch``      many systems with several right-hand sides each, solved together.

Matrices come from the library's generator (NPB's makea).  Orders, nonzeros per vector and shifts
are the NPB classes' own or follow the range the shipped network was trained on,
shift = (nonzer + 1)^2 * [0.3, 0.45], where every system is definite.
"""
import math
import os
import random
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "npb-gpu_amd"))
import npbcg  # noqa: E402

RTOL = 1e-10
CG_STEPS = 25        # inner steps of conj_grad
SOLVE_STEPS = 8      # CG steps a solve of this family needs to 1e-10 (kappa about 1.4)
NET_FILE = os.path.join(ROOT, "npb-gpu_amd", "npbcg", "learned_precond.npz")
MODES = {"fp64": npbcg.SOLVE_FP64, "mixed": npbcg.SOLVE_MIXED}
PRECONDS = {"none": npbcg.PRECOND_NONE, "jacobi": npbcg.PRECOND_JACOBI,
            "neumann": npbcg.PRECOND_NEUMANN}


def listed():
    return [
        # NPB class S: the smallest run, 375 CG steps on a matrix of 78 thousand entries
        {"name": "power_n1400", "kind": "power", "n": 1400, "nonzer": 7, "shift": 10.0,
         "niter": 15},
        # NPB class A
        {"name": "power_n14000", "kind": "power", "n": 14000, "nonzer": 11, "shift": 20.0,
         "niter": 15},
        # NPB class B, the benchmark's workload: a matrix that fits the memory-side cache
        {"name": "power_n75000", "kind": "power", "n": 75000, "nonzer": 13, "shift": 60.0,
         "niter": 75},
        # NPB class C: a matrix larger than that cache; the largest case
        {"name": "power_n150000", "kind": "power", "n": 150000, "nonzer": 15, "shift": 110.0,
         "niter": 75},
        # a program that swaps the serial conj_grad for the library's, arrays on the host
        {"name": "conj_grad_n30011", "kind": "conj_grad", "n": 30011, "nonzer": 10,
         "shift": 45.0},
        # a small system kept on the GPU, one FP64 solve after another (a time step's solves)
        {"name": "solve_fp64_n7001", "kind": "solve", "n": 7001, "nonzer": 8, "shift": 30.0,
         "mode": "fp64", "precond": "none", "nrhs": 4},
        # the solve of the headline comparison: mixed precision at the largest order
        {"name": "solve_mixed_n150000", "kind": "solve", "n": 150000, "nonzer": 15,
         "shift": 110.0, "mode": "mixed", "precond": "none", "nrhs": 4},
        # one system, solved once: layout and upload are part of what the caller waits for
        {"name": "oneoff_fp64_n30011", "kind": "oneoff", "n": 30011, "nonzer": 10,
         "shift": 45.0, "mode": "fp64"},
        # the learned preconditioner in use: inference for the matrix, then two solves
        {"name": "learned_mixed_n60013", "kind": "learned", "n": 60013, "nonzer": 12,
         "shift": 60.0, "nrhs": 2},
        # one training step's forward and backward on a system of the training range
        {"name": "train_grad_n40009", "kind": "train_grad", "n": 40009, "nonzer": 11,
         "shift": 52.0, "pairs": 8},
        # a batch of ragged systems in mixed precision with four right-hand sides
        {"name": "batch_mixed_16x4", "kind": "batch", "systems": 16, "nrhs": 4, "mode": "mixed",
         "n_min": 2000, "n_max": 40000},
        # a handful of small systems in FP64, one right-hand side: too few rows to fill the GPU
        {"name": "batch_fp64_6x1", "kind": "batch", "systems": 6, "nrhs": 1, "mode": "fp64",
         "n_min": 2000, "n_max": 8000},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _family(rng, n):
    """nonzer and shift for order n: denser rows for larger systems, as the NPB classes."""
    top = 15 if n >= 60000 else 13
    nonzer = rng.randint(7, top)
    return nonzer, round((nonzer + 1) ** 2 * rng.uniform(0.3, 0.45), 3)


def draw(rng):
    kind = rng.choice(["power", "power", "power", "conj_grad", "solve", "solve", "solve",
                       "oneoff", "learned", "train_grad", "batch", "batch"])
    c = {"kind": kind}
    if kind == "batch":
        lo = _log_int(rng, 1000, 6000)
        c.update(systems=_log_int(rng, 2, 20), nrhs=rng.choice([1, 2, 4]),
                 mode=rng.choice(["fp64", "mixed"]), n_min=lo,
                 n_max=_log_int(rng, lo + 500, 40000))
        return c
    lo, hi = {"power": (1400, 150000), "conj_grad": (1400, 75000), "solve": (1400, 150000),
              "oneoff": (2000, 75000), "learned": (17000, 75000),
              "train_grad": (10000, 75000)}[kind]
    n = _log_int(rng, lo, hi)
    c["n"] = n
    c["nonzer"], c["shift"] = _family(rng, n)
    if kind == "power":
        c["niter"] = rng.randint(5, 40)
    elif kind == "solve":
        # mixed precision needs the LDS-staged layout, the library's choice from 16384 rows up
        c["mode"] = rng.choice(["fp64", "mixed"]) if n >= 17000 else "fp64"
        c["precond"] = rng.choice(["none", "none", "jacobi", "neumann"])
        c["nrhs"] = rng.randint(1, 6)
    elif kind == "oneoff":
        c["mode"] = rng.choice(["fp64", "mixed"]) if n >= 17000 else "fp64"
    elif kind == "learned":
        c["nrhs"] = rng.randint(1, 4)
    elif kind == "train_grad":
        c["pairs"] = rng.randint(4, 8)
    return c


# ---- inputs -----------------------------------------------------------------------------------


def _lcg_seed(seed):
    """An NPB generator seed (an odd integer below 2^46) that follows from `seed`."""
    return float(random.Random(seed).randrange(1 << 20, 1 << 45) | 1)


def _matrix(case, seed):
    return npbcg.makea(case["n"], case["nonzer"], case["shift"], _lcg_seed(seed))


def _vectors(case, seed, count):
    rng = np.random.default_rng([seed, 1])
    return [rng.uniform(-1.0, 1.0, case["n"]) for _ in range(count)]


def _batch_systems(case, seed):
    """Orders spread evenly over the range (shuffled, so ragged in order too) and per-system
    nonzer; the sizes are the case's, the matrices and right-hand sides the seed's."""
    k, lo, hi = case["systems"], case["n_min"], case["n_max"]
    shape = random.Random(k * 1000003 + lo * 31 + hi)
    ns = [lo + (hi - lo) * i // max(1, k - 1) for i in range(k)]
    shape.shuffle(ns)
    out = []
    for i, n in enumerate(ns):
        nonzer = shape.randint(7, 13)
        out.append((n, nonzer, (nonzer + 1) ** 2 * shape.uniform(0.3, 0.45),
                    _lcg_seed(seed * 1009 + i), 0.1))
    return out


def _batch_rhs(case, seed, systems):
    rng = np.random.default_rng([seed, 2])
    return [rng.uniform(-1.0, 1.0, (s[0], case["nrhs"])) for s in systems]


def _net_params():
    with np.load(NET_FILE, allow_pickle=False) as f:
        return f["params"].copy(), f["norm"].copy()


def _train_params(seed):
    """Parameters in the middle of training: the shipped ones, disturbed."""
    params, norm = _net_params()
    rng = np.random.default_rng([seed, 3])
    return (params + 0.05 * rng.standard_normal(params.size)).astype(np.float32), norm


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind == "batch":
        systems = _batch_systems(case, seed)
        mats = npbcg.make_many(systems)
        s["batch"] = npbcg.Batch(mats, nrhs=case["nrhs"], mode=MODES[case["mode"]])
        s["rhs"] = _batch_rhs(case, seed, systems)
        return s
    s["m"] = _matrix(case, seed)
    if kind == "oneoff":
        s["b"] = _vectors(case, seed, 1)[0]
        return s
    s["ctx"] = npbcg.Context(s["m"])
    if kind == "conj_grad":
        # the reference calls it on the normalised iterate; any vector of that scale
        s["x"] = np.append(_vectors(case, seed, 1)[0], 0.0)
    elif kind == "solve":
        s["ctx"].set_preconditioner(PRECONDS[case["precond"]])
        s["b"] = _vectors(case, seed, case["nrhs"])
    elif kind == "learned":
        s["net"] = npbcg.Net()
        s["net"].load(NET_FILE)
        s["b"] = _vectors(case, seed, case["nrhs"])
    elif kind == "train_grad":
        s["net"] = npbcg.Net()
        s["net"].set_params(*_train_params(seed))
        s["ctx"].set_rhs(_vectors(case, seed, 1)[0])
        s["ctx"].log_pairs(case["pairs"])
    return s


# ---- one pass ---------------------------------------------------------------------------------


def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "power":
        ctx = s["ctx"]
        ctx.fill_x(1.0)
        zeta, rnorm = ctx.power(c["niter"], c["shift"])
        # the table a run prints, one row an iteration (rnorm is at rounding level), and the
        # eigenvector it leaves
        return {"table": np.stack([zeta, rnorm]), "x": ctx.get_vector(npbcg.VEC_X)}
    if kind == "conj_grad":
        z, p, q, r, rnorm = s["ctx"].conj_grad(s["x"])
        # the vectors as the call leaves them, side by side: p, q and rnorm are what rounding
        # leaves of them after 25 steps
        return np.concatenate([z, p, q, r, [rnorm]])
    if kind == "solve":
        out = []
        for b in s["b"]:
            s["ctx"].set_rhs(b)
            s["ctx"].solve(MODES[c["mode"]], RTOL, 500)
            out.append(s["ctx"].solution())
        return out
    if kind == "oneoff":
        with npbcg.Context(s["m"]) as ctx:
            ctx.set_rhs(s["b"])
            ctx.solve(MODES[c["mode"]], RTOL, 500)
            return ctx.solution()
    if kind == "learned":
        ctx = s["ctx"]
        s["net"].apply(ctx)
        ctx.set_preconditioner(npbcg.PRECOND_LEARNED)
        out = []
        for b in s["b"]:
            ctx.set_rhs(b)
            ctx.solve(npbcg.SOLVE_MIXED, RTOL, 500)
            out.append(ctx.solution())
        return out
    if kind == "train_grad":
        loss, grad, gh = s["net"].loss_grad(s["ctx"], c["n"])
        return {"loss": loss, "grad": grad, "gh": gh}
    s["batch"].set_rhs(s["rhs"])
    s["batch"].solve(RTOL, 500)
    return np.concatenate([x.reshape(-1) for x in s["batch"].solution()])


# ---- the work a pass cannot do without ---------------------------------------------------------


def _nnz(n, nonzer):
    """Entries of the generator's matrix (expected): the diagonal, and the off-diagonals of n outer
    products of nonzer + 1 entries less the positions that coincide."""
    full = n * (nonzer + 1) * nonzer
    return n + n * n * -math.expm1(-full / (n * n))


def _spmv(n, nonzer, value=8):
    """Bytes and operations of one product: the CSR (values of `value` bytes, 4-byte columns,
    row pointers) and the vector read, the result written."""
    nnz = _nnz(n, nonzer)
    return nnz * (value + 4) + 4 * (n + 1) + 2 * value * n, 2.0 * nnz


def work(case):
    kind = case["kind"]
    if kind == "batch":
        b = f = 0.0
        for n, nonzer, *_ in _batch_systems(case, 0):
            w = {"n": n, "nonzer": nonzer, "mode": case["mode"], "kind": "solve", "nrhs": 1}
            one, k = work(w), case["nrhs"]
            vec = SOLVE_STEPS * 72.0 * n
            b += one["bytes"] + (k - 1) * vec  # the matrices are read once for all vectors
            f += k * one["flops"]
        return {"bytes": b, "flops": f}
    n, nonzer = case["n"], case["nonzer"]
    b64, f1 = _spmv(n, nonzer)
    b32, _ = _spmv(n, nonzer, 4)
    if kind in ("power", "conj_grad"):
        it = case.get("niter", 1)
        b = it * ((CG_STEPS + 1) * b64 + CG_STEPS * 72.0 * n + 56.0 * n)
        f = it * ((CG_STEPS + 1) * f1 + CG_STEPS * 10.0 * n)
        return {"bytes": b, "flops": f}
    if kind == "train_grad":
        # forward and backward of a 32-64 embedding and three 128-64 layers per row (the weights
        # stay on chip): the rows' features, graph and pairs in, g, h and the gradient out
        gemm = 32 * 64 + 3 * 128 * 64
        p = case["pairs"]
        return {"bytes": n * (8 * 4 + 4 * 12 + 8 + 8.0 * p + 8) + 4.0 * 27010,
                "flops": 6.0 * n * gemm + n * p * 80.0}
    mixed = kind == "learned" or case["mode"] == "mixed"
    if mixed:  # FP32 steps, and an FP64 residual in each of two sweeps
        b = (SOLVE_STEPS + 1) * (b32 + 36.0 * n) + 2 * (b64 + 24.0 * n)
        f = (SOLVE_STEPS + 3) * f1
    else:
        b = SOLVE_STEPS * (b64 + 72.0 * n) + b64 + 24.0 * n
        f = (SOLVE_STEPS + 1) * f1
    k = 1 if kind == "oneoff" else case["nrhs"]
    b, f = k * b, k * f
    if kind == "learned":
        b += n * (8 * 4 + 4 * 8 + 8.0)
        f += 2.0 * n * (32 * 64 + 3 * 128 * 64)
    return {"bytes": b, "flops": f}


# ---- the same values in plain 64-bit torch -----------------------------------------------------

DEV = "cuda" if torch.cuda.is_available() else "cpu"


def _product(m):
    a = torch.sparse_csr_tensor(torch.from_numpy(m.rowstr.astype(np.int64)),
                                torch.from_numpy(m.colidx.astype(np.int64)),
                                torch.from_numpy(m.a), size=(m.n, m.n)).to(DEV)
    return lambda v: a @ v


def _cg(mul, b, steps=None, log=0):
    """CG from x = 0: `steps` steps, or until the residual stops falling (steps = None).
    With log > 0 also the first `log` pairs of residual and iterate."""
    x, r = torch.zeros_like(b), b.clone()
    p, rho = r.clone(), float(r @ r)
    pairs, tol = [], 1e-30 * rho
    for k in range(steps if steps is not None else 400):
        if len(pairs) < log:
            pairs.append((r.clone(), x.clone()))
        if steps is None and rho <= tol:
            break
        q = mul(p)
        alpha = rho / float(p @ q)
        x = x + alpha * p
        r = r - alpha * q
        rho, old = float(r @ r), rho
        if rho == 0.0:
            break
        p = r + (rho / old) * p
    return x, pairs


def _exact_solution(m, b):
    mul = _product(m)
    b = torch.from_numpy(np.ascontiguousarray(b)).to(DEV)
    x, _ = _cg(mul, b)
    return (x + _cg(mul, b - mul(x))[0]).cpu().numpy()


def _exact_grad(case, seed):
    m = _matrix(case, seed)
    n, K, H = m.n, 4, 64
    t = lambda v, dt=torch.float64: torch.as_tensor(np.ascontiguousarray(v)).to(DEV, dt)  # noqa: E731
    length = t(np.diff(m.rowstr), torch.int64)
    row = torch.repeat_interleave(torch.arange(n, device=DEV), length)
    col, a = t(m.colidx, torch.int64), t(m.a)
    diag = torch.zeros(n, dtype=torch.float64, device=DEV)
    diag[row[row == col]] = a[row == col]
    # features and the four largest off-diagonals of every row (largest first, ties by column)
    off = row != col
    orow, ocol, oa = row[off], col[off], a[off]
    ad, av = diag.abs(), oa.abs()
    sums = lambda v: torch.zeros(n, dtype=torch.float64, device=DEV).index_add_(0, orow, v)  # noqa: E731
    top = torch.zeros(n, dtype=torch.float64, device=DEV).scatter_reduce_(0, orow, av, "amax")
    dk = ad[ocol]
    feat = torch.stack([sums(av) / ad, sums(oa * oa) / ad ** 2, top / ad, sums(oa) / ad,
                        sums(oa * oa / (ad[orow] * dk)), sums(av / (ad[orow] * dk).sqrt()),
                        torch.log2(length.double()) / 8.0, torch.log10(ad) / 3.0], dim=1)
    by = torch.argsort(av, descending=True, stable=True)
    by = by[torch.argsort(orow[by], stable=True)]
    first = torch.cumsum(torch.bincount(orow, minlength=n), 0) - torch.bincount(orow, minlength=n)
    pick = by[(first[:, None] + torch.arange(K, device=DEV))]
    nbr, val = ocol[pick], oa[pick]
    w = val.abs() / (ad[:, None] * ad[nbr]).sqrt()
    w = w / w.sum(1, keepdim=True)
    nval = val / (diag[:, None] * diag[nbr])
    # the pairs: residuals of CG from 0 and the corrections still missing
    mul = _product(m)
    b = t(_vectors(case, seed, 1)[0])
    xs, pairs = _cg(mul, b, log=case["pairs"])
    params, norm = _train_params(seed)
    p, norm = t(params).requires_grad_(True), t(norm)
    x = torch.zeros(n, 32, dtype=torch.float64, device=DEV)
    x[:, :8] = (feat - norm[:8]) / norm[8:]
    at = 0

    def take(*shape):
        nonlocal at
        k = math.prod(shape)
        at += k
        return p[at - k:at].reshape(shape)

    w0, b0 = take(32, H), take(H)
    h = torch.relu(x @ w0 + b0)
    for _ in range(3):
        wl, bl = take(2 * H, H), take(H)
        agg = sum(w[:, k:k + 1] * h[nbr[:, k]] for k in range(K))
        h = torch.relu(torch.cat([h, agg], 1) @ wl + bl)
    ug, cg, uh, ch = take(H), take(1), take(H), take(1)
    g, hh = torch.tanh(h @ ug + cg), torch.tanh(h @ uh + ch)
    q = torch.exp(g + hh)

    def both(v):
        out = (nval * v[nbr]).sum(1)
        return out.index_add(0, nbr.reshape(-1), (nval * v[:, None]).reshape(-1))

    loss = 0.0
    for r, xk in pairs:
        e = xs - xk
        y = torch.exp(2 * g) / diag * r - q * both(q * r)
        loss = loss + ((y - e) ** 2).sum() / (len(pairs) * (e * e).sum())
    loss.backward()
    return {"loss": loss.item(), "grad": p.grad.cpu().numpy(),
            "gh": torch.cat([g, hh]).detach().cpu().numpy()}


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        systems = _batch_systems(case, seed)
        out = []
        for m, b in zip(npbcg.make_many(systems), _batch_rhs(case, seed, systems)):
            x = np.stack([_exact_solution(m, b[:, k]) for k in range(case["nrhs"])], axis=1)
            out.append(x.reshape(-1))
        return np.concatenate(out)
    if kind == "train_grad":
        return _exact_grad(case, seed)
    m = _matrix(case, seed)
    if kind == "power":
        mul = _product(m)
        x = torch.ones(m.n, dtype=torch.float64, device=DEV)
        zeta, rnorm = [], []
        for _ in range(case["niter"]):
            z, _ = _cg(mul, x, CG_STEPS)
            zeta.append(case["shift"] + 1.0 / float(x @ z))
            rnorm.append(float((x - mul(z)).norm()))
            x = z / z.norm()
        return {"table": np.array([zeta, rnorm]), "x": np.append(x.cpu().numpy(), 1.0)}
    if kind == "conj_grad":
        x = _vectors(case, seed, 1)[0]
        z = _exact_solution(m, x)
        nil = np.zeros(m.n + 1)
        # 25 steps converge to rounding: z solves A z = x, r = A z, and p, q, ||x - A z|| vanish;
        # index n holds x[n] = 0 in all of them
        return np.concatenate([np.append(z, 0.0), nil, nil, np.append(x, 0.0), [0.0]])
    count = 1 if kind == "oneoff" else case["nrhs"]
    out = [_exact_solution(m, b) for b in _vectors(case, seed, count)]
    return out[0] if kind == "oneoff" else out
