"""The blocked Cholesky with its fused forward substitution, through the weight
fit, at the sizes where its panels change: less than one panel, whole panels,
one column more, and a matrix that starts with a super-panel (more than 4096
columns).  The fit's solution is held to its own optimality conditions with
the gradient and residual of separate kernels: A^T (1 - A x) vanishes on the
active set (bar 1e-8 of the largest |A^T 1|: the normal equations of these
well-conditioned fits leave 1e-13, an unsolved column of order 1).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [30, 63, 64, 65, 127, 128, 129, 191, 192, 193, 320, 333, 1000, 4096, 4161, 4353])
def test_fit_is_optimal(oracle, n):
    import numcosmo_amd as na
    d = 12
    g = np.random.default_rng(n)
    X = g.normal(size=(n, d))
    m2lnp = np.sum(X * X, axis=1)
    sd = na.StatsDistVKDE.new(na.StatsDistKernelST.new(d, 3.0), na.StatsDistCV.NONE)
    sd.set_local_frac(max(0.05, 20.0 / n))
    sd.add_obs_array(X)
    sd.prepare_interp(m2lnp)
    x, grad, r = sd.peek_nnls_state()
    rungs = sd.get_nnls_rungs()
    assert rungs[0] >= 1 and rungs[1] == 0 and rungs[2] == 0
    act = x > 0.0
    assert act.sum() > n // 2
    A = sd.compute_IM() / np.exp(-0.5 * (m2lnp - m2lnp.min()))[:, None]
    scale = np.max(A.sum(axis=0))
    assert np.max(np.abs(grad[act])) < 1e-8 * scale
    assert np.max(np.abs(r - (1.0 - A @ x))) < 1e-10
    assert np.all(grad[~act] < 1e-8 * scale)
    if n <= 400:
        od = oracle.StatsDist(1, 1, d, 3.0)
        od.set_local_frac(max(0.05, 20.0 / n))
        od.add_obs_array(X)
        od.prepare_interp(m2lnp)
        w, wo = sd.peek_weights(), od.get_weights()
        assert np.abs(w - wo).sum() < 1e-9 * np.abs(wo).sum()
