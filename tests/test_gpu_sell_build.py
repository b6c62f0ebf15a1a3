"""The SELL copy as the device builds it: at the edges of blocks, ranges, sort
windows and slices the stored entries (padding included) are those of the
layout's definition, computed here from the CSR, and q = A p, conj_grad and a
mixed solve on it match the oracle (1e-12 relative; solutions 1e-8)."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def _stored(rowstr, colidx, n, W, R, window):
    total = 0
    row = np.repeat(np.arange(n), np.diff(rowstr))
    for b in range(-(-n // W)):
        inside = (colidx >= b * W) & (colidx < (b + 1) * W)
        length = np.bincount(row[inside], minlength=n)
        for r0 in range(0, n, R):
            part = length[r0:min(n, r0 + R)]
            for w0 in range(0, part.size, window):
                s = -np.sort(-part[w0:w0 + window], kind="stable")
                total += 64 * int(s[::64].sum())
    return total


def _matrix(gpu, n, k, seed):
    """Random symmetric diagonally dominant CSR in which every third row has
    its diagonal only."""
    import scipy.sparse as sp

    rng = np.random.default_rng(seed)
    rows, cols = rng.integers(0, n, n * k), rng.integers(0, n, n * k)
    keep = (rows != cols) & (rows % 3 != 1) & (cols % 3 != 1)
    up = sp.coo_matrix((rng.uniform(-1, 1, n * k)[keep], (rows[keep], cols[keep])),
                       shape=(n, n)).tocsr()
    off = (up + up.T).tocsr()
    m = (off + sp.diags(np.asarray(abs(off).sum(axis=1)).ravel() + 1.0)).tocsr()
    m.sort_indices()
    rs, ci, a = m.indptr.astype(np.int32), m.indices.astype(np.int32), m.data.copy()
    return gpu.Matrix(n, rs, ci, a), oracle.CSR(n, rs, ci, a, 1.0, 0, 10.0, 0.1, float(seed))


@pytest.mark.parametrize("n,width,rows,window", [
    (1, 0, 0, 0),
    (65, 2, 64, 64),           # many blocks of two columns
    (4097, 1000, 4096, 0),     # a last range of one row
    (5000, 5000, 63, 64),      # ranges shorter than a slice
    (9001, 3002, 2049, 2048),  # a window of one row at the end of every range
    (20011, 0, 0, 0),
    (20011, 7000, 9000, 8192),   # the widest window the device sorts
    (20011, 7000, 20011, 16384), # wider: built on the host
])
def test_layout_and_results(gpu, n, width, rows, window):
    m, om = _matrix(gpu, n, 9, seed=n + width)
    x = np.append(np.random.default_rng(3).uniform(-1, 1, n), [2.0, 0.0])
    b = np.random.default_rng(4).uniform(-1, 1, n)
    with gpu.Context(m, spmv_variant=5, tile_width=width, tile_rows=rows,
                     sort_window=window) as ctx:
        d = ctx.describe()
        assert d["spmv_variant"] == 5
        assert d["sell_stored"] == _stored(m.rowstr, m.colidx, n, d["block_width"],
                                           d["range_rows"], d["sort_window"])
        if n > 2:   # 25 fixed steps divide 0 by 0 at orders 1 and 2
            z, p, q, r, rn = ctx.conj_grad(x)
            for v, ref in zip((z, p, q, r), oracle.conj_grad(om, x)):
                assert np.max(np.abs(v[:n] - ref[:n])) <= 1e-12 * max(1.0, np.max(np.abs(ref)))
        ctx.set_rhs(b)
        assert ctx.solve(gpu.SOLVE_MIXED, 1e-10, 500).converged == 1
        s = ctx.solution()
    ox, _, _ = oracle.cg_solve(om, b, rtol=1e-10, maxit=1000)
    assert np.max(np.abs(s - ox)) <= 1e-8 * np.max(np.abs(ox))


def test_columns_are_checked_on_the_device(gpu):
    m, _ = _matrix(gpu, 3000, 5, seed=1)
    for k, v in ((17, 3000), (m.nnz - 1, -1)):
        ci = m.colidx.copy()
        ci[k] = v
        with pytest.raises(gpu.NpbcgError) as e:
            gpu.Context(gpu.Matrix(m.n, m.rowstr, ci, m.a))
        assert e.value.code == gpu.ERR_INVALID
