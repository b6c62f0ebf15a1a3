"""A launch of the resident engine that gives up waiting: whichever launch of a call it is,
the call's results are bit for bit those of the kernels engine, from the x it was given, and
for a while no context of the process tries that engine again."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RESIDENT, KERNELS = 2, 1   # npbcg_timing.engine


def _give_up(gpu, ctx, iteration):
    assert gpu.LIB.npbcg_test_resident_give_up(ctx._h, iteration) == 0, gpu.last_error()


@pytest.fixture(autouse=True)
def _rested(gpu):
    yield
    with gpu.Context(gpu.makea(1400, 7, 10.0, 271.0)) as ctx:
        _give_up(gpu, ctx, -1)   # the tests that follow use the engine again


@pytest.mark.parametrize("iteration", [0, 17, 33])   # launches of 16, 16 and 2 iterations
def test_power_loop(gpu, iteration):
    m = gpu.makea(19000, 7, 20.0, 271.0)
    x = np.random.default_rng(1).uniform(0.5, 1.0, m.n + 1)
    with gpu.Context(m, engine=KERNELS) as ctx:
        ctx.set_vector(gpu.VEC_X, x)
        want = (*ctx.power(34, 20.0), ctx.get_vector(gpu.VEC_X))
    with gpu.Context(m) as ctx:
        ctx.set_vector(gpu.VEC_X, x)
        _give_up(gpu, ctx, 34)   # past the last: nothing gives up
        ctx.power(34, 20.0)
        assert ctx.timing().engine == RESIDENT
        ctx.set_vector(gpu.VEC_X, x)
        _give_up(gpu, ctx, iteration)
        got = (*ctx.power(34, 20.0), ctx.get_vector(gpu.VEC_X))
        assert ctx.timing().engine == KERNELS
    for u, v in zip(got, want):
        assert np.array_equal(u, v)


def test_profile(gpu):
    m = gpu.makea(19000, 7, 20.0, 271.0)
    with gpu.Context(m, engine=KERNELS) as ctx:
        want = ctx.profile_kernels(20, 20.0)
    with gpu.Context(m) as ctx:
        _give_up(gpu, ctx, 0)
        got = ctx.profile_kernels(20, 20.0)
    assert np.array_equal(got[2], want[2])
    assert [k["name"] for k in got[0]] == [k["name"] for k in want[0]]


def test_conj_grad_and_solve(gpu):
    m = gpu.makea(7001, 8, 30.0, 271.0)
    rng = np.random.default_rng(2)
    x, b = rng.uniform(-1, 1, m.n + 1), rng.uniform(-1, 1, m.n)

    def calls(ctx):
        return (*ctx.conj_grad(x), ctx.get_vector(gpu.VEC_X))

    def solve(ctx):
        ctx.set_rhs(b)
        st = ctx.solve(gpu.SOLVE_FP64, 1e-10, 500)
        return ctx.solution(), st.iterations, st.relres, st.converged

    with gpu.Context(m, engine=KERNELS) as ctx:
        want, want_solve = calls(ctx), solve(ctx)
    with gpu.Context(m) as ctx:
        _give_up(gpu, ctx, 0)
        got = calls(ctx)
        assert ctx.timing().engine == KERNELS
    with gpu.Context(m) as ctx:
        _give_up(gpu, ctx, 0)
        got_solve = solve(ctx)
    for u, v in zip(got + got_solve, want + want_solve):
        assert np.array_equal(u, v)


def test_other_contexts_do_not_wait_too(gpu):
    m = gpu.makea(1400, 7, 10.0, 271.0)
    x = np.random.default_rng(3).uniform(-1, 1, m.n + 1)
    with gpu.Context(m) as first, gpu.Context(m) as second:
        want = second.conj_grad(x)
        assert second.timing().engine == RESIDENT
        _give_up(gpu, first, 0)
        first.conj_grad(x)
        with gpu.Context(m) as third:
            for ctx in (first, second, third):
                ctx.conj_grad(x)
                assert ctx.timing().engine == KERNELS
            _give_up(gpu, first, -1)   # the rest is over
            for ctx in (first, second, third):
                got = ctx.conj_grad(x)
                assert ctx.timing().engine == RESIDENT
                for u, v in zip(got, want):
                    assert np.array_equal(u, v)
