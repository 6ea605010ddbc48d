"""Fits that end with an error: what they refuse, and the handle afterwards."""
import numpy as np
import pytest

from numcosmo_amd._lib import NckdeError

pytestmark = pytest.mark.gpu

EINVAL, ENUMERIC = -1, -7


def _new(kind, kernel, d, umethod=0):
    import numcosmo_amd as na
    k = na.StatsDistKernelGauss.new(d) if kernel == 0 else na.StatsDistKernelST.new(d, 3.0)
    sd = (na.StatsDistVKDE if kind == 1 else na.StatsDistKDE).new(k)
    if kind == 1:
        sd.set_local_frac(0.3)
    sd.set_nnls_umethod(umethod)
    return sd


@pytest.mark.parametrize("umethod", [0, 1, 2], ids=["NORMAL", "NORMAL_LU", "QR"])
@pytest.mark.parametrize("n", [32, 65, 200])
def test_nan_m2lnp(umethod, n):
    """A NaN in m2lnp makes every entry of the normal matrix NaN: each rung
    fails, the fit ends with the error of a total weight that is not positive,
    and the handle takes a good fit afterwards.  n = 32 and 65: the matrix ends
    where its buffer ends, so that a pivot index of n would be out of range."""
    g = np.random.default_rng(n)
    X = g.normal(size=(n, 3))
    m2 = np.sum(X * X, 1)
    bad = m2.copy()
    bad[n // 2] = np.nan
    sd = _new(1, 1, 3, umethod)
    sd.add_obs_array(X)
    with pytest.raises(NckdeError) as e:
        sd.prepare_interp(bad)
    assert e.value.status == ENUMERIC
    sd.prepare_interp(m2)
    twin = _new(1, 1, 3, umethod)
    twin.add_obs_array(X)
    twin.prepare_interp(m2)
    assert np.array_equal(sd.peek_weights(), twin.peek_weights())


def test_refused_length_leaves_uniform_weights():
    """m2lnp of the wrong length: the sample is prepared, with equal weights,
    and they are there when the call returns, also while other work holds the
    GPU (the getter reads on another stream than the prepare writes on)."""
    import torch
    from numcosmo_amd._lib import lib
    g = np.random.default_rng(7)
    n, d = 600, 4
    X = g.normal(size=(n, d))
    m2 = np.sum(X * X, 1)
    sd = _new(0, 0, d)
    sd.add_obs_array(X)
    A = torch.randn(4096, 4096, device="cuda")
    side = torch.cuda.Stream()
    for _ in range(20):
        sd.prepare_interp(m2)
        w = np.empty(n)
        assert not np.allclose(sd.peek_weights(), 1.0 / n)
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            for _ in range(10):
                A @ A
        assert lib().nckde_prepare_interp(sd._h, np.append(m2, 0.0), n + 1) == EINVAL
        assert lib().nckde_get_weights(sd._h, w) == 0
        assert np.array_equal(w, np.full(n, 1.0 / n))
    torch.cuda.synchronize()


@pytest.mark.parametrize("kind,kernel", [(0, 0), (1, 1), (1, 0)])
@pytest.mark.parametrize("why", ["nan", "zero"])
def test_no_positive_weight_keeps_the_prepared_density(kind, kernel, why):
    """A fit whose weights have no positive total (NaN in m2lnp; a bandwidth so
    wide that every kernel underflows to 0) ends with an error, and the handle
    evaluates as its prepare left it, with equal weights, in every precision."""
    g = np.random.default_rng(9)
    n, d = 300, 3
    X = g.normal(size=(n, d))
    m2 = np.sum(X * X, 1)
    P = g.normal(size=(3000, d))
    sd, twin = _new(kind, kernel, d), _new(kind, kernel, d)
    for o in (sd, twin):
        if why == "zero":
            o.set_over_smooth(1e110)
        o.add_obs_array(X)
    if why == "nan":
        m2[n // 2] = np.nan
    with pytest.raises(NckdeError) as e:
        sd.prepare_interp(m2)
    assert e.value.status == ENUMERIC
    twin.prepare()
    for precision in (0, 1, 2):
        got, ref = sd.eval_m2lnp_batch(P, precision), twin.eval_m2lnp_batch(P, precision)
        assert np.all(np.isfinite(ref))
        assert np.array_equal(got, ref)
