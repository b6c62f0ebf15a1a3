"""The resident engine (small orders, everything left to the library) on the
GPU: conj_grad, the power loop and FP64 solves at the edges of its kernels'
ranges against the oracle, with the tolerances of the other engines' tests
(vectors and zeta 1e-12 relative, solutions 1e-8); columns in any order; rows
longer than the registers hold, and rows too long for it; a power loop of
several launches; calls of two contexts from two threads."""
import threading

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

RESIDENT, KERNELS = 2, 1   # npbcg_timing.engine


def _matrix(gpu, n, k, seed, shuffle=False, arrow=False):
    """Random symmetric diagonally dominant CSR: about 2 k off-diagonals a row,
    with `arrow` a full first row and column of small entries."""
    import scipy.sparse as sp

    rng = np.random.default_rng(seed)
    rows = np.repeat(np.arange(n), k)
    cols = rng.integers(0, n, size=n * k)
    if arrow:
        rows = np.concatenate([rows, np.zeros(n - 1, int)])
        cols = np.concatenate([cols, np.arange(1, n)])
    vals = rng.uniform(-1.0, 1.0, size=rows.size)
    if arrow:  # light enough for 25 steps to converge
        vals[n * k:] *= 0.002
    keep = rows != cols
    up = sp.coo_matrix((vals[keep], (rows[keep], cols[keep])), shape=(n, n)).tocsr()
    off = (up + up.T).tocsr()
    d = np.asarray(abs(off).sum(axis=1)).ravel() + 1.0
    m = (off + sp.diags(d)).tocsr()
    m.sort_indices()
    rs, ci, a = m.indptr.astype(np.int32), m.indices.astype(np.int32), m.data.copy()
    if shuffle:
        for j in range(n):
            s, e = rs[j], rs[j + 1]
            perm = s + rng.permutation(e - s)
            ci[s:e], a[s:e] = ci[perm].copy(), a[perm].copy()
    return gpu.Matrix(n, rs, ci, a), oracle.CSR(n, rs, ci, a, 1.0, 0, 10.0, 0.1, float(seed))


def _close(v, ref, scale, label):
    err = float(np.max(np.abs(v - ref)))
    assert err <= 1e-12 * max(1.0, scale, float(np.max(np.abs(ref)))), f"{label}: {err:.3e}"


def _check(gpu, m, om, engine, niter=2):
    n = m.n
    rng = np.random.default_rng(n)
    x = rng.uniform(-1.0, 1.0, n + 2)
    x[n] = 3.0
    b = rng.uniform(-1.0, 1.0, n)
    with gpu.Context(m) as ctx:
        z, p, q, r, rn = ctx.conj_grad(x)
        assert ctx.timing().engine == engine
        oz, op, oq, orr, orn = oracle.conj_grad(om, x)
        for v, ref, lab in ((z, oz, "z"), (p, op, "p"), (q, oq, "q"), (r, orr, "r")):
            _close(v[:n], ref[:n], 1.0, f"n={n} {lab}")
        assert abs(rn - orn) <= 1e-12 * np.linalg.norm(x[:n])
        assert z[n] == 0.0 and q[n] == 0.0 and r[n] == 3.0 and p[n] == 3.0
        ctx.fill_x(1.0)
        zeta, rnorm = ctx.power(niter, om.shift)
        ozeta, ornorm, _ = oracle.power(om, niter)
        assert np.max(np.abs(zeta - ozeta) / np.abs(ozeta)) <= 1e-12, n
        assert np.max(np.abs(rnorm - ornorm)) <= 1e-12 * np.sqrt(n), n
        xs = ctx.get_vector(gpu.VEC_X)[:n]
        assert abs(np.linalg.norm(xs) - 1.0) <= 1e-12
        ctx.set_rhs(b)
        st = ctx.solve(gpu.SOLVE_FP64, 1e-10, 500)
        s = ctx.solution()
    assert st.converged == 1 and np.linalg.norm(b - oracle.spmv(om, s)) <= 1e-10 * np.linalg.norm(b)
    ox, _, _ = oracle.cg_solve(om, b, rtol=1e-10, maxit=1000)
    assert np.max(np.abs(s - ox)) <= 1e-8 * np.max(np.abs(ox))


# the last order of each kernel and the first of the next; 19153 is the first
# the engine leaves to the others
@pytest.mark.parametrize("n", [3, 15, 16, 1920, 1921, 3840, 3841, 7936, 7937, 16128, 16129,
                               19152, 19153])
def test_orders_at_the_edges(gpu, n):
    m, om = _matrix(gpu, n, min(12, n), seed=n)
    _check(gpu, m, om, RESIDENT if n <= 19152 else KERNELS)


@pytest.mark.parametrize("n,k,shuffle,arrow,engine", [
    (900, 300, False, False, RESIDENT),   # dense rows: past the registers' entries
    (6000, 120, True, False, RESIDENT),   # columns in any order
    (12000, 2, True, False, RESIDENT),    # a few entries a row
    (1900, 5, False, True, RESIDENT),     # one row of 1900 entries
    (5000, 5, False, True, KERNELS),      # one row longer than its lanes take
])
def test_row_lengths(gpu, n, k, shuffle, arrow, engine):
    m, om = _matrix(gpu, n, k, seed=n + k, shuffle=shuffle, arrow=arrow)
    _check(gpu, m, om, engine)


def test_power_in_several_launches(gpu):
    # 16 outer iterations fill the exchange workspace at this order
    m, om = _matrix(gpu, 19152, 6, seed=4)
    _check(gpu, m, om, RESIDENT, niter=18)


def test_two_threads(gpu):
    mats = [gpu.makea(7000, 8, 12.0, 1.0 + s) for s in (2, 4)]
    ctxs = [gpu.Context(m) for m in mats]
    want = [c.power(4, 12.0) for c in ctxs]
    got = [[], []]

    def run(i):
        for _ in range(5):
            ctxs[i].fill_x(1.0)
            got[i].append(ctxs[i].power(4, 12.0))

    ts = [threading.Thread(target=run, args=(i,)) for i in (0, 1)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for i in (0, 1):
        assert len(got[i]) == 5 and ctxs[i].timing().engine == RESIDENT
        for z, r in got[i]:
            assert np.array_equal(z, want[i][0]) and np.array_equal(r, want[i][1])
        ctxs[i].close()
