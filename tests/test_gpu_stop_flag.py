"""A solve's stop test is made by every workgroup of the kernel that updates p, and recorded by
one of them while others may be reading the flag.  Whichever they find, no workgroup updates
p after the last step: one solve after another leaves the same bits of p and of the solution
(the SELL kernel with the update inside, the separate update, sparse preconditioners)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,kw", [(9001, {"spmv_variant": 3}), (17003, {}), (49153, {}),
                                  (45000, {"spmv_variant": 5})])
@pytest.mark.parametrize("precond", [0, 1, 3])
def test_p_after_the_last_step(gpu, n, kw, precond):
    m = gpu.makea(n, 9, 38.0, 271.0)
    b = np.random.default_rng(n).uniform(-1, 1, n)
    with gpu.Context(m, engine=1, **kw) as ctx:
        ctx.set_preconditioner(precond)
        ctx.set_rhs(b)
        first = None
        for i in range(60):
            st = ctx.solve(gpu.SOLVE_FP64, 1e-10, 500)
            if i < 2:   # the first solve has another number of launches
                continue
            got = (ctx.get_vector(gpu.VEC_P)[:n], ctx.solution(), st.iterations)
            first = first or got
            for u, v in zip(got, first):
                assert np.array_equal(u, v), (n, precond, i)


def test_batch_after_the_last_step(gpu):
    orders = [300 + 700 * i for i in range(24)]
    mats = gpu.make_many([(n, 7, 22.0, 1001.0 + 2 * n) for n in orders])
    rng = np.random.default_rng(3)
    b = [rng.uniform(-1, 1, (n, 2)) * 10.0 ** rng.integers(-6, 6, 2) for n in orders]
    with gpu.Batch(mats, nrhs=2, mode=0) as bt:
        bt.set_rhs(b)
        first = None
        for _ in range(40):
            st, steps, rel = bt.solve(1e-10, 500)
            got = [steps, rel, *bt.solution()]
            first = first or got
            for u, v in zip(got, first):
                assert np.array_equal(u, v)
