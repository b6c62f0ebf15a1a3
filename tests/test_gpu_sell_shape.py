"""The default shape of the SELL copy: six column blocks while the LDS would
hold the vector in fewer, ranges of whole 64-row slices, eight wavefronts up to
16 slices; conj_grad and a mixed solve at the edges of the rule match the
oracle (1e-12 relative; solutions 1e-8)."""
import numpy as np
import pytest

import oracle
from test_gpu_sell_build import _matrix

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,blocks,rows,threads", [
    (96, 6, 64, 512),            # 16 columns a block
    (2688, 6, 64, 512),          # 42 ranges of one slice
    (2689, 6, 128, 512),         # a last range of one row
    (43008, 6, 1024, 512),       # 16 slices
    (43009, 6, 1088, 1024),      # 17 slices
    (120000, 6, 2880, 1024),
    (121344, 7, None, 1024),     # six of the widest blocks leave the LDS no room for slots
])
def test_default_shape(gpu, n, blocks, rows, threads):
    m, om = _matrix(gpu, n, 9, seed=n)
    x = np.append(np.random.default_rng(3).uniform(-1, 1, n), [2.0, 0.0])
    b = np.random.default_rng(4).uniform(-1, 1, n)
    with gpu.Context(m, spmv_variant=5, engine=1) as ctx:
        d = ctx.describe()
        assert (d["col_blocks"], d["sell_threads"]) == (blocks, threads)
        assert rows is None or d["range_rows"] == rows
        assert (d["block_width"] + (d["range_rows"] + 63) // 64) * 8 <= 160 * 1024
        z, p, q, r, rn = ctx.conj_grad(x)
        ctx.set_rhs(b)
        assert ctx.solve(gpu.SOLVE_MIXED, 1e-10, 500).converged == 1
        s = ctx.solution()
    ref = oracle.conj_grad(om, x)[0]
    assert np.max(np.abs(z[:n] - ref[:n])) <= 1e-12 * max(1.0, np.max(np.abs(ref)))
    ox, _, _ = oracle.cg_solve(om, b, rtol=1e-10, maxit=1000)
    assert np.max(np.abs(s - ox)) <= 1e-8 * np.max(np.abs(ox))
