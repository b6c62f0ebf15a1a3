"""The network's (g, h) where its 16-row tiles and wavefronts end, from a pass that keeps
its activations (loss and gradient) and one that does not (inference).  (g, h) against the
oracle within the BF16 activations' rounding (2e-2: a few BF16 ulps of outputs of order 1);
the operator that inference installs against the dense M^-1 of the kept pass's (g, h),
where both hold the same float32 values: 1e-12."""
import numpy as np
import pytest

import oracle
from oracle import learned as ol

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [15, 16, 17, 31, 33, 127, 129, 1025])
def test_network_at_tile_edges(gpu, n):
    m = gpu.makea(n, 3 if n < 100 else 6, 6.0 if n < 100 else 20.0, 91.0)
    g = ol.graph(oracle.CSR(n, m.rowstr, m.colidx, m.a, m.ratio, m.nonzer, m.shift, m.rcond, m.seed))
    g.nval = g.nval.astype(np.float32).astype(np.float64)   # the device keeps N in float32
    norm = ol.feature_norm(g)
    rng = np.random.default_rng(n)
    params = (rng.standard_normal(ol.N_PARAMS) * 0.15).astype(np.float32)
    params[ol.OFF_W0 + ol.F * ol.H:ol.OFF_B0] = 0.0
    r, e = (rng.standard_normal((2, n)).astype(np.float32) for _ in range(2))
    v = rng.standard_normal(n)
    with gpu.Context(m, spmv_variant=1) as ctx, gpu.Net(seed=3) as net:
        net.set_params(params, norm)
        net.apply(ctx)                       # first: nothing kept from another pass
        ctx.set_preconditioner(gpu.PRECOND_LEARNED)
        z = ctx.apply_preconditioner(v)
        ctx.set_pairs(r, e)
        _, _, gh = net.loss_grad(ctx, n)
    _, _, wgh = ol.loss_and_grad(params.astype(np.float64), norm, g, r.astype(np.float64),
                                 e.astype(np.float64), bf16_on=True)
    assert np.max(np.abs(gh - wgh)) <= 2e-2, np.max(np.abs(gh - wgh))
    want = ol.precond_dense(g, gh.astype(np.float64)) @ v
    assert np.allclose(z, want, rtol=1e-12, atol=1e-14 * np.max(np.abs(want)))
