"""No memory for the buffers of the resident engine: the calls run on the kernels engine with
its bits, whichever buffer is missing, and on the resident one again once there is memory."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RESIDENT, KERNELS = 2, 1   # npbcg_timing.engine


def _calls(gpu, c, b):
    """Results of a power loop of 40 iterations (two launches), conj_grad and a solve."""
    out, engines = [], []
    c.fill_x(1.0)
    out += [*c.power(40, 20.0), c.get_vector(gpu.VEC_X)]
    engines.append(c.timing().engine)
    out += [c.conj_grad_device(), c.get_vector(gpu.VEC_Z)]
    engines.append(c.timing().engine)
    c.set_rhs(b)
    c.solve(gpu.SOLVE_FP64, 1e-10, 500)
    out.append(c.solution())
    _, _, zeta = c.profile_kernels(3, 20.0)
    return out + [zeta], engines


@pytest.mark.parametrize("warm", [False, True])   # nothing there yet; buffers too small
def test_no_memory(gpu, warm):
    m = gpu.makea(17000, 7, 20.0, 271.0)
    b = np.random.default_rng(3).uniform(-1, 1, m.n)
    with gpu.Context(m, engine=KERNELS) as c:
        want, _ = _calls(gpu, c, b)
    with gpu.Context(m) as c:
        if warm:
            c.fill_x(1.0)
            c.power(1, 20.0)
            assert c.timing().engine == RESIDENT
        assert gpu.LIB.npbcg_test_no_memory(c._h, 1) == 0
        c.fill_x(1.0)
        got = [*c.power(40, 20.0), c.get_vector(gpu.VEC_X)]
        assert c.timing().engine == KERNELS
        for u, v in zip(got, want):
            assert np.array_equal(u, v)
        if not warm:
            got, engines = _calls(gpu, c, b)
            assert engines == [KERNELS, KERNELS]
            for u, v in zip(got, want):
                assert np.array_equal(u, v)
        assert gpu.LIB.npbcg_test_no_memory(c._h, 0) == 0
        assert _calls(gpu, c, b)[1] == [RESIDENT, RESIDENT]
