"""FP64 solves that come again replay a captured graph up to the orders where launching is
as fast, on the CSR kernels and on the SELL copy (p update fused and apart): the bits of
launched ones, with other right-hand sides and calls in between."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _band(gpu, n, half):
    """Symmetric band of 2 half + 1 entries a row (wrapped around), diagonally dominant."""
    o = np.concatenate([np.arange(-half, half + 1)])
    col = (np.arange(n)[:, None] + o) % n
    a = np.where(o == 0, 2.0 * half + 1.0, -1.0 / (1 + np.abs(o)))
    order = np.argsort(col, axis=1)
    col = np.take_along_axis(col, order, axis=1)
    a = np.take_along_axis(np.broadcast_to(a, col.shape), order, axis=1)
    rs = (np.arange(n + 1) * (2 * half + 1)).astype(np.int32)
    return gpu.Matrix(n, rs, col.reshape(-1).astype(np.int32), a.reshape(-1).copy())


@pytest.mark.parametrize("kind,n", [("csr", 16384), ("csr", 131071), ("csr", 131072),
                                    ("sell", 16500), ("sell", 32767), ("sell", 32768),
                                    ("wide", 25000)])
def test_replays_are_the_launches(gpu, kind, n):
    m = (_band(gpu, n, 2) if kind == "csr" else _band(gpu, n, 40) if kind == "wide"
         else gpu.makea(n, 7, 22.0, 271.0))
    rng = np.random.default_rng(n)
    b = [rng.uniform(-1, 1, n) for _ in range(2)]
    x = rng.uniform(-1, 1, n + 1)
    with gpu.Context(m, engine=1) as ctx, gpu.Context(m, engine=1, use_graph=0) as plain:
        assert (ctx.describe()["spmv_variant"] == 5) == (kind != "csr")
        for i in range(18):
            got = []
            for c in (ctx, plain):
                c.set_preconditioner((gpu.PRECOND_JACOBI, gpu.PRECOND_NEUMANN,
                                      gpu.PRECOND_NONE)[i // 6])
                c.set_rhs(b[i % 2])
                st = c.solve(gpu.SOLVE_FP64, 1e-10, 500)
                got.append((c.solution(), st.iterations, st.relres, st.sweeps))
                if i % 5 == 4:
                    c.conj_grad(x)
            for u, v in zip(*got):
                assert np.array_equal(u, v), (n, i)
            if i % 6 == 5:   # each preconditioner's sequence was seen six times
                captured = gpu.LIB.npbcg_test_solve_graphs(ctx._h)
                assert (captured > 0) == (n < (131072 if kind == "csr" else 32768)), (n, i)
        assert gpu.LIB.npbcg_test_solve_graphs(plain._h) == 0
