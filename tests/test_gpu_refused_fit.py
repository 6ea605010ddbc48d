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
