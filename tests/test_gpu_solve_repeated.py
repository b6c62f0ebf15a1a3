"""FP64 solves that come again on the CSR kernels replay a captured graph from the fourth
on: every solve gives the bits of launched ones, with other right-hand sides,
preconditioners, tolerances and calls of other kinds between the replays."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [300, 4001, 16383, 16384])
def test_replays_are_the_launches(gpu, n):
    m = gpu.makea(n, 7, 22.0, 271.0)
    rng = np.random.default_rng(n)
    b = [rng.uniform(-1, 1, n) for _ in range(3)]
    x = rng.uniform(-1, 1, n + 1)
    with gpu.Context(m, engine=1, spmv_variant=3) as ctx, \
            gpu.Context(m, engine=1, spmv_variant=3, use_graph=0) as plain:
        for i in range(36):
            precond = (gpu.PRECOND_JACOBI, gpu.PRECOND_NEUMANN, gpu.PRECOND_NONE)[i // 6 % 3]
            rtol = 1e-10 if i % 12 < 9 else 1e-6
            got = []
            for c in (ctx, plain):
                c.set_preconditioner(precond)
                c.set_rhs(b[0 if i < 24 else i % 3])
                st = c.solve(gpu.SOLVE_FP64, rtol, 500)
                got.append((c.solution(), st.iterations, st.relres, st.sweeps))
                if i % 5 == 4:
                    c.conj_grad(x)
            for u, v in zip(*got):
                assert np.array_equal(u, v), (n, i)
