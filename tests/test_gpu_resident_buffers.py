"""Solves and power loops in turn on one context of the resident engine, whose exchange
buffers and partial sums grow by themselves: every call gives the bits of the first round,
from either order of first calls."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [3, 2000, 19152])
def test_solve_and_power_in_turn(gpu, n):
    m = gpu.makea(n, 7 if n > 3 else 1, 15.0 if n > 3 else 1.0, 271.0)
    b = np.random.default_rng(0).uniform(-1, 1, n)

    def solve(c):
        c.solve(gpu.SOLVE_FP64, 1e-10, 500)
        return (c.solution(),)

    def power(c, niter):   # 26 exchanges and a set of partials an iteration; a solve 65 and one
        c.fill_x(1.0)
        return c.power(niter, 15.0)

    with gpu.Context(m) as first, gpu.Context(m) as second:
        for c in (first, second):
            c.set_rhs(b)
        want = (solve(first), power(first, 2), power(first, 17))
        for c in (second, first, second):
            for niter in (17, 2, 17):
                for got, ref in ((power(c, niter), want[1 if niter == 2 else 2]),
                                 (solve(c), want[0])):
                    for u, v in zip(got, ref):
                        assert np.array_equal(u, v, equal_nan=True)
