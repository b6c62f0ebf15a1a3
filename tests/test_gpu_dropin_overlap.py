"""The drop-in call digests the caller's arrays while the GPU works: a call whose arrays
differ is refused and leaves the context's vectors, scalars and timing bit for bit as they
were (the resident, SELL and CSR engines), and the next good call gives the bits of the
first."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,kw", [(1, {}), (1400, {}), (30011, {}), (3001, {"spmv_variant": 3})])
def test_refused_call_changes_nothing(gpu, n, kw):
    if n == 1:
        m = gpu.Matrix(1, np.array([0, 1], np.int32), np.array([0], np.int32), np.array([2.5]))
    else:
        m = gpu.makea(n, 7, 20.0, 271.0)
    rng = np.random.default_rng(n)
    x, y = rng.uniform(-1, 1, n + 1), rng.uniform(-1, 1, n + 1)
    with gpu.Context(m, **kw) as ctx:
        first = ctx.conj_grad(x)
        before = [ctx.get_vector(w) for w in range(5)]
        timing = bytes(ctx.timing())
        for array, change in ((m.a, 1.0), (m.colidx, 1)):
            k = m.nnz - 1
            saved = array[k]
            array[k] += change
            try:
                with pytest.raises(gpu.NpbcgError) as e:
                    ctx.conj_grad(y)
                assert e.value.code == gpu.ERR_MISMATCH
            finally:
                array[k] = saved
            for w, v in enumerate(before):
                assert np.array_equal(ctx.get_vector(w), v, equal_nan=True), w
            assert bytes(ctx.timing()) == timing
        again = ctx.conj_grad(x)
        for u, v in zip(first, again):
            assert np.array_equal(u, v, equal_nan=True)
