"""A drop-in call with another matrix of the same rows is refused before any work is done
for it, by the samples, and the context stays as it was; the compat call goes on to the other
matrix."""
import ctypes
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_refused_before_the_work(gpu):
    m = gpu.makea(30011, 10, 45.0, 271.0)
    other = 1.5 * m.a
    x = np.random.default_rng(0).uniform(-1, 1, m.n + 1)
    good, refused = [], []
    with gpu.Context(m) as ctx:
        ctx.conj_grad(x)
        before = [ctx.get_vector(w) for w in range(5)]
        for _ in range(20):
            t = time.perf_counter()
            ctx.conj_grad(x)
            good.append(time.perf_counter() - t)
            t = time.perf_counter()
            with pytest.raises(gpu.NpbcgError) as e:
                ctx.conj_grad(x, a=other)
            refused.append(time.perf_counter() - t)
            assert e.value.code == gpu.ERR_MISMATCH
        for w, v in enumerate(before):
            assert np.array_equal(ctx.get_vector(w), v), w
    assert np.median(refused) <= 0.5 * np.median(good), (refused, good)


def test_compat_call_takes_the_other_matrix(gpu):
    m = gpu.makea(3001, 7, 20.0, 271.0)
    x = np.random.default_rng(1).uniform(-1, 1, m.n + 1)
    with gpu.Context(gpu.Matrix(m.n, m.rowstr, m.colidx, 1.5 * m.a)) as ctx:
        want = ctx.conj_grad(x)
    assert gpu.LIB.npbcg_compat_set_n(m.n) == 0
    try:
        for a in (m.a, 1.5 * m.a):
            z, p, q, r = (np.zeros(m.n + 1) for _ in range(4))
            rn = ctypes.c_double(0.0)
            gpu.LIB.npbcg_compat_conj_grad(m.colidx, m.rowstr, x, z, a, p, q, r, ctypes.byref(rn))
    finally:
        gpu.LIB.npbcg_compat_release()
    for u, v in zip((z, p, q, r, rn.value), want):
        assert np.array_equal(u, v)
