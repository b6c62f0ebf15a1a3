"""Solves whose steps update p inside the SpMV (every FP32 step; FP64 up to order 49152,
apart past it): an odd last column of a block, one slice, both sides of that order, with
every kind of preconditioner.  True residuals formed here in FP64 meet the tolerance, and
the reported ones are those (1e-13 of ||b|| for another order of summation)."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [65, 97, 4099, 49152, 49153])
@pytest.mark.parametrize("precond", [0, 1, 3])
@pytest.mark.parametrize("mode", [0, 1])
def test_fused_p_update(gpu, n, precond, mode):
    m = gpu.makea(n, 3 if n < 100 else 7, 6.0 if n < 100 else 22.0, 100.0 + n)
    a = sp.csr_matrix((m.a, m.colidx, m.rowstr), shape=(n, n))
    rng = np.random.default_rng(n)
    with gpu.Context(m, spmv_variant=5, engine=1) as ctx:
        ctx.set_preconditioner(precond)
        for _ in range(2):
            b = rng.uniform(-1, 1, n)
            ctx.set_rhs(b)
            st = ctx.solve(mode, 1e-10, 500)
            true = np.linalg.norm(b - a @ ctx.solution()) / np.linalg.norm(b)
            assert st.converged and true <= 1e-10 + 1e-13
            assert abs(true - st.relres) <= 1e-13
