"""The resident engine at the last order of each of its kernels and the first of the
next: conj_grad and an FP64 solve against the oracle (1e-12 relative; solutions 1e-8)."""
import numpy as np
import pytest

import oracle
from test_gpu_resident import RESIDENT, _close, _matrix

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [960, 961, 1440, 1441, 2400, 2401, 2880, 3361, 4960, 4961, 5953, 6944,
                               6945, 9072, 9073, 10081, 11088, 12097, 13104, 14113, 15121, 17136,
                               17137, 18145])
def test_every_kernel(gpu, n):
    m, om = _matrix(gpu, n, 12, seed=n)
    rng = np.random.default_rng(n)
    x = np.append(rng.uniform(-1.0, 1.0, n), [3.0, 0.0])
    b = rng.uniform(-1.0, 1.0, n)
    with gpu.Context(m) as ctx:
        got = ctx.conj_grad(x)
        assert ctx.timing().engine == RESIDENT
        for v, ref, name in zip(got, oracle.conj_grad(om, x), "zpqr"):
            _close(v[:n], ref[:n], float(np.max(np.abs(x))), f"n {n} {name}")
        ctx.set_rhs(b)
        assert ctx.solve(gpu.SOLVE_FP64, 1e-10, 500).converged == 1
        s = ctx.solution()
    ox, _, _ = oracle.cg_solve(om, b, rtol=1e-10, maxit=1000)
    assert np.max(np.abs(s - ox)) <= 1e-8 * np.max(np.abs(ox))
