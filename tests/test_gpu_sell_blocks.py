"""Column blocks of the default SELL copy, by the matrix: the widest that fit where a row's
entries lie in one or two blocks (bands, stencils) or the rows are short and alike, six
where they are anywhere in a row (makea).  conj_grad and a mixed solve match the oracle
(1e-12 relative; solutions 1e-8)."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def _offsets(kind, n):
    if kind == "band":
        return np.arange(1, 41)
    if kind == "stencil":   # 27 points of a cube of side s
        s = round(n ** (1 / 3))
        o = {abs(x + s * y + s * s * z) for x in (-1, 0, 1) for y in (-1, 0, 1) for z in (-1, 0, 1)}
        return np.array(sorted(o - {0}))
    if kind == "spread":    # 40 entries over the whole row
        return np.arange(1, 21) * (n // 41) + 3
    return np.arange(1, 8)  # 15 entries: below the library's own choice of this layout


def _matrix(gpu, kind, n):
    """A symmetric circulant pattern with random values, diagonally dominant."""
    import scipy.sparse as sp

    rng = np.random.default_rng(n)
    i = np.arange(n)
    up = sum(sp.coo_matrix((rng.uniform(-1, 1, n), (i, (i + o) % n)), shape=(n, n))
             for o in _offsets(kind, n)).tocsr()
    off = (up + up.T).tocsr()
    m = (off + sp.diags(np.asarray(abs(off).sum(axis=1)).ravel() + 1.0)).tocsr()
    m.sort_indices()
    rs, ci, a = m.indptr.astype(np.int32), m.indices.astype(np.int32), m.data.copy()
    return gpu.Matrix(n, rs, ci, a), oracle.CSR(n, rs, ci, a, 1.0, 0, 10.0, 0.1, float(n))


@pytest.mark.parametrize("kind,n,blocks", [
    ("band", 20000, 1), ("band", 25000, 2), ("band", 48001, 3), ("band", 97003, 5),
    ("stencil", 48001, 3), ("spread", 48001, 3),
    ("few", 48001, 6), ("band", 121068, 6),
])
def test_blocks_follow_the_matrix(gpu, kind, n, blocks):
    m, om = _matrix(gpu, kind, n)
    x = np.append(np.random.default_rng(3).uniform(-1, 1, n), [2.0, 0.0])
    b = np.random.default_rng(4).uniform(-1, 1, n)
    with gpu.Context(m, spmv_variant=5, engine=1) as ctx:
        assert ctx.describe()["col_blocks"] == blocks
        z, p, q, r, rn = ctx.conj_grad(x)
        ctx.set_rhs(b)
        assert ctx.solve(gpu.SOLVE_MIXED, 1e-10, 500).converged == 1
        s = ctx.solution()
    ref = oracle.conj_grad(om, x)[0]
    assert np.max(np.abs(z[:n] - ref[:n])) <= 1e-12 * max(1.0, np.max(np.abs(ref)))
    ox, _, _ = oracle.cg_solve(om, b, rtol=1e-10, maxit=1000)
    assert np.max(np.abs(s - ox)) <= 1e-8 * np.max(np.abs(ox))


@pytest.mark.parametrize("n,nonzer", [(20000, 7), (30011, 10), (75000, 13), (97003, 7)])
def test_six_for_makea(gpu, n, nonzer):
    with gpu.Context(gpu.makea(n, nonzer, (nonzer + 1) ** 2 * 0.38, 271.0), engine=1) as ctx:
        assert ctx.describe()["col_blocks"] == 6
