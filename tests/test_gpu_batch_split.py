"""Batches of few rows: their sorting windows are short and a slice's entries are
shared by several wavefronts.  From one 64-row window to several windows per CU,
ragged at the ends of windows and slices, the solutions' true residuals, formed
here from the CSR in FP64, meet the tolerance, and the reported ones are those
(rounding of a residual formed in another order: 1e-13 of ||b||)."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("orders,nrhs,mode", [
    ((65,), 1, 0),
    ((64, 20, 63, 129), 2, 0),
    ((2048, 2049), 4, 1),
    ((9001, 2000), 4, 1),
    ((3000, 16511, 30000), 2, 0),
    (tuple(range(2000, 20000, 950)), 1, 1),
    (tuple(range(4000, 36000, 4500)), 4, 0),
])
def test_split_windows(gpu, orders, nrhs, mode):
    rng = np.random.default_rng(len(orders))
    mats = gpu.make_many([(n, 7 if n > 100 else 3, 25.0 if n > 100 else 6.0, 1001.0 + 2 * n)
                          for n in orders])
    b = [rng.uniform(-1, 1, (n, nrhs)) for n in orders]
    with gpu.Batch(mats, nrhs=nrhs, mode=mode, layout=3) as bt:
        for _ in range(2):
            bt.set_rhs(b)
            st, steps, rel = bt.solve(1e-10, 500)
            x = bt.solution()
    assert st.converged == st.solves == len(orders) * nrhs
    for m, bs, xs, rs in zip(mats, b, x, rel):
        a = sp.csr_matrix((m.a, m.colidx, m.rowstr), shape=(m.n, m.n))
        true = np.linalg.norm(bs - a @ xs, axis=0) / np.linalg.norm(bs, axis=0)
        assert np.all(true <= 1e-10 + 1e-13), (m.n, true)
        assert np.all(np.abs(true - rs) <= 1e-13), (m.n, true, rs)
