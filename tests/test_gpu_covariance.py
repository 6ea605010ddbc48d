"""Global and local covariances against the oracle's one-pass recurrence, bit
for bit, at the edges of the kernel's 2 x 2 entry tiles (odd and even
dimensions) and of its row chunks (2048 / d rows for the global matrix, 512 / d
and more for the local ones)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,n,lf", [(1, 40, 0.3), (2, 1025, 0.3), (3, 683, 0.9), (5, 410, 0.9), (16, 128, 0.5),
                                    (16, 129, 0.26), (17, 241, 0.5), (31, 133, 0.9), (32, 64, 0.9), (63, 99, 0.9),
                                    (64, 160, 0.9)])
def test_covariances_bit_exact(oracle, d, n, lf):
    import numcosmo_amd as na
    g = np.random.default_rng(d * n)
    X = g.normal(size=(n, d)) * 10.0 ** g.uniform(-2, 2, size=d) + g.normal(size=d)
    X[1] = X[0]                      # a zero difference in the recurrence
    sd = na.StatsDistVKDE.new(na.StatsDistKernelGauss.new(d), na.StatsDistCV.NONE)
    od = oracle.StatsDist(1, 0, d, 0.0)
    for o in (sd, od):
        o.set_local_frac(lf)
        o.add_obs_array(X)
        o.prepare()
    assert np.array_equal(sd.peek_full_cov(), od.get_full_cov())
    for i in (0, 1, n // 2, n - 1):
        assert np.array_equal(np.triu(sd.peek_cov_decomp(i)), np.triu(od.get_cov_decomp(i)))
