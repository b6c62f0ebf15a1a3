"""Resident launches of several contexts follow one another on the GPU while their callers
do not wait for each other's host work: results as when called alone, beside drop-in calls
that hash a large matrix while their launch runs, and when a context whose launch was the
last is destroyed."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RESIDENT = 2   # npbcg_timing.engine


def _band(gpu, n, half):
    """A symmetric band matrix of 2 half + 1 diagonals, diagonally dominant."""
    j = np.arange(n)[:, None] + np.arange(-half, half + 1)[None, :]
    keep = (j >= 0) & (j < n)
    d = np.abs(np.arange(-half, half + 1))
    v = np.where(d == 0, 2.0 * half, 1.0 / (1.0 + d))
    rowstr = np.concatenate([[0], np.cumsum(keep.sum(1))]).astype(np.int32)
    return gpu.Matrix(n, rowstr, j[keep].astype(np.int32),
                      np.broadcast_to(v, j.shape)[keep].astype(np.float64))


def test_calls_beside_hashing_ones(gpu):
    big, small = _band(gpu, 18000, 200), gpu.makea(1400, 7, 10.0, 271.0)
    x = np.random.default_rng(0).uniform(-1, 1, 18001)
    with gpu.Context(big) as a, gpu.Context(small) as b:
        want, alone = a.conj_grad(x), b.power(2, 10.0)
        assert a.timing().engine == RESIDENT and b.timing().engine == RESIDENT
        calls = []

        def hashing():
            for _ in range(40):
                calls.append(a.conj_grad(x))

        th = threading.Thread(target=hashing)
        th.start()
        while th.is_alive():
            b.fill_x(1.0)
            for u, v in zip(b.power(2, 10.0), alone):
                assert np.array_equal(u, v)
        th.join()
    assert len(calls) == 40
    for got in calls:
        for u, v in zip(got, want):
            assert np.array_equal(u, v)


def test_contexts_come_and_go(gpu):
    mats = [gpu.makea(n, 7, 15.0, 271.0) for n in (1400, 5000, 9000, 19000)]
    rng = np.random.default_rng(1)
    b = [rng.uniform(-1, 1, m.n) for m in mats]
    want = []
    for m, v in zip(mats, b):
        with gpu.Context(m) as ctx:
            ctx.set_rhs(v)
            ctx.solve(gpu.SOLVE_FP64, 1e-10, 500)
            want.append((ctx.solution(), *ctx.power(3, 15.0)))
    bad = []

    def run(i):
        for _ in range(8):
            with gpu.Context(mats[i]) as ctx:
                ctx.set_rhs(b[i])
                ctx.solve(gpu.SOLVE_FP64, 1e-10, 500)
                got = (ctx.solution(), *ctx.power(3, 15.0))
                if not all(np.array_equal(u, v) for u, v in zip(got, want[i])):
                    bad.append(i)

    ts = [threading.Thread(target=run, args=(i,)) for i in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
