"""The drop-in call without memory to keep the context's state in: the same results, and an
edited matrix is refused before any work."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1400, 30011])
def test_drop_in_without_memory(gpu, n):
    m = gpu.makea(n, 7, 20.0, 271.0)
    rng = np.random.default_rng(n)
    x, y = rng.uniform(-1, 1, n + 1), rng.uniform(-1, 1, n + 1)
    with gpu.Context(m, engine=1) as ctx:
        want = ctx.conj_grad(x)
    with gpu.Context(m, engine=1) as ctx:
        assert gpu.LIB.npbcg_test_no_memory(ctx._h, 1) == 0
        first = ctx.conj_grad(x)
        for u, v in zip(first, want):
            assert np.array_equal(u, v)
        before = [ctx.get_vector(w) for w in range(5)]
        value = m.a[1]
        m.a[1] += 1.0   # between the samples
        try:
            with pytest.raises(gpu.NpbcgError) as e:
                ctx.conj_grad(y)
            assert e.value.code == gpu.ERR_MISMATCH
        finally:
            m.a[1] = value
        for w, v in enumerate(before):
            assert np.array_equal(ctx.get_vector(w), v), w
