"""The two forms of the FP64 per-pair terms (a power of an inverse square root
or 2^t against a common reference; ln K with an online maximum) and the merge
of the split sums, against the FP64 oracle at the sizes where they change:
integer and non-integer nu, the largest power taken, dimensions around the
padded ones, points whose terms underflow, and point counts around the block
and merge layouts.  Bar: 1e-12 relative (the terms' rounding, |ln K| ulps of
each, averages below 1e-14; the bar of the other FP64 eval tests).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _pair(oracle, kind, nu, d, X):
    import numcosmo_amd as na
    sdk = na.StatsDistKernelGauss.new(d) if nu == 0.0 else na.StatsDistKernelST.new(d, nu)
    sd = (na.StatsDistVKDE if kind == 1 else na.StatsDistKDE).new(sdk, na.StatsDistCV.NONE)
    od = oracle.StatsDist(kind, 0 if nu == 0.0 else 1, d, nu)
    for o in (sd, od):
        if kind == 1:
            o.set_local_frac(0.4)
        o.add_obs_array(X)
        o.prepare()
    return sd, od


def _check(sd, od, P):
    got, ref = sd.eval_m2lnp_batch(P, 0), od.eval_m2lnp_batch(P)
    assert np.max(np.abs(got - ref) / np.maximum(np.abs(ref), 1.0)) < 1e-12


@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("nu", [0.0, 1.0, 2.0, 2.5, 3.0])
@pytest.mark.parametrize("d", [1, 3, 4, 5, 6, 7, 12, 13, 15, 16, 17, 20, 21, 24, 25, 29, 33, 37, 48, 49, 53, 57, 64])
def test_forms_by_dimension(oracle, kind, nu, d):
    g = np.random.default_rng(d)
    n = 3 * d + 40
    X = g.normal(size=(n, d))
    sd, od = _pair(oracle, kind, nu, d, X)
    P = np.concatenate([X[:5], g.normal(size=(60, d)), 30.0 * g.normal(size=(5, d))])
    _check(sd, od, P)


@pytest.mark.parametrize("nu", [122.0, 123.0, 124.0, 0.0, 5.0])
def test_largest_power_and_underflow(oracle, nu):
    """nu + d = 126, 127 (fast), 128 (general); far points whose terms all
    underflow against the common reference."""
    g = np.random.default_rng(3)
    X = g.normal(size=(200, 4))
    sd, od = _pair(oracle, 1, nu, 4, X)
    P = np.concatenate([g.normal(size=(50, 4)) * s for s in (1.0, 1e2, 1e5, 1e9)])
    _check(sd, od, P)


@pytest.mark.parametrize("nu", [0.0, 2.5, 3.0])
@pytest.mark.parametrize("d", [5, 16, 33])
def test_non_finite_points(oracle, nu, d):
    """A point with NaN or inf has density 0 (m2lnp = +inf) and leaves the
    points beside it alone."""
    g = np.random.default_rng(4)
    X = g.normal(size=(160, d))
    sd, od = _pair(oracle, 1, nu, d, X)
    P = g.normal(size=(70, d))
    clean = sd.eval_m2lnp_batch(P, 0)
    Q = P.copy()
    Q[3, 0] = np.nan
    Q[17, d - 1] = np.inf
    Q[69, d // 2] = -np.inf
    got = sd.eval_m2lnp_batch(Q, 0)
    bad = [3, 17, 69]
    assert np.all(np.isposinf(got[bad]))
    keep = np.setdiff1d(np.arange(70), bad)
    assert np.array_equal(got[keep], clean[keep])


@pytest.mark.parametrize("m", [1, 2, 63, 64, 65, 128, 129, 255, 257, 2047, 2048, 2049])
@pytest.mark.parametrize("d", [3, 16, 40])
@pytest.mark.parametrize("precision", [0, 2])
def test_point_counts(oracle, m, d, precision):
    g = np.random.default_rng(m)
    X = g.normal(size=(333, d))
    sd, od = _pair(oracle, 1, 3.0, d, X)
    P = g.normal(size=(m, d))
    got, ref = sd.eval_m2lnp_batch(P, precision), od.eval_m2lnp_batch(P)
    assert np.max(np.abs(got - ref) / np.maximum(np.abs(ref), 1.0)) < (1e-12 if precision == 0 else 1e-6)


@pytest.mark.parametrize("nu", [0.0, 2.5, 3.0])
@pytest.mark.parametrize("d,n", [(5, 70), (12, 257), (13, 64), (16, 129), (17, 300), (24, 320), (36, 333), (64, 515)])
def test_interpolation_matrix(oracle, nu, d, n):
    """IM of the vector and the matrix-core forms: kernels and observations
    that leave partial tiles.  1e-11: chi2 reaches 1e3 on the outer pairs and
    ln K turns its 1e-15 relative error into 1e-12 of K."""
    g = np.random.default_rng(d + n)
    X = g.normal(size=(n, d))
    sd, od = _pair(oracle, 1, nu, d, X)
    got, ref = sd.compute_IM(), od.compute_IM()
    assert np.max(np.abs(got - ref) / np.maximum(np.abs(ref), 1e-300)) < 1e-11


@pytest.mark.parametrize("nu", [0.0, 3.0])
@pytest.mark.parametrize("d,n", [(2, 1601), (3, 1604), (4, 1607), (5, 1601), (8, 1603), (9, 1601), (12, 1602),
                                 (16, 1601), (16, 1603), (17, 1601), (32, 1603), (33, 1601), (48, 1603), (49, 1601),
                                 (64, 1603)])
def test_mixed_groups(oracle, nu, d, n):
    """Mixed evals with kernel counts that leave part of a group (8, 4, 4, 2, 2
    kernels), and point counts around the 32-point tiles and the blocks of 512
    (768 at d = 9 to 16): 1e-6 relative, the bar of the mixed path.  More than 800
    points of 1600 kernels, since fewer run in FP64."""
    g = np.random.default_rng(d * n)
    X = g.normal(size=(n, d))
    sd, od = _pair(oracle, 1, nu, d, X)
    # the probe of the riskiest kernels (1e-6 at d = 64) would send the handle to FP64
    sd.set_mixed_tolerance(1e-5)
    assert not sd.get_mixed_check()[1]
    P = np.concatenate([g.normal(size=(1601, d)), X[:1], 40.0 * g.normal(size=(1, d))])
    ref = od.eval_m2lnp_batch(P)
    for m in (800, 801, 831, 1024, 1025, 1536, 1537, 1603):
        Q, r = P[-m:], ref[-m:]
        got = sd.eval_m2lnp_batch(Q, 1)
        # the mixed form ran: the FP64 one gives the FP64 eval's results to the bit
        assert not np.array_equal(got, sd.eval_m2lnp_batch(Q, 0))
        assert np.max(np.abs(got - r) / np.maximum(np.abs(r), 1.0)) < 1e-6


@pytest.mark.parametrize("d", [3, 7])
@pytest.mark.parametrize("extra", [-1, 0, 1])
def test_host_staging(oracle, d, extra):
    """Host-buffer evals around the size (256 KiB of points and results) up to
    which they go through the pinned buffer, packed and with a row stride: each
    point's value does not depend on the way it came in."""
    import numcosmo_amd as na
    from numcosmo_amd._lib import check, lib
    g = np.random.default_rng(8)
    X = g.normal(size=(120, d))
    sd, od = _pair(oracle, 1, 3.0, d, X)
    m = (256 << 10) // (8 * (d + 1)) + extra
    wide = g.normal(size=(m, d + 2))
    P = np.ascontiguousarray(wide[:, :d])
    got = sd.eval_m2lnp_batch(P, 0)
    out = np.empty(m)
    check(lib().nckde_eval_m2lnp(sd._h, wide, m, d + 2, out, 0))
    assert np.array_equal(got, out)
    ref = od.eval_m2lnp_batch(P[-50:])
    assert np.max(np.abs(got[-50:] - ref) / np.maximum(np.abs(ref), 1.0)) < 1e-12
    # a smaller call afterwards reuses the buffer
    assert np.max(np.abs(sd.eval_m2lnp_batch(P[:5], 0) - got[:5]) / np.maximum(np.abs(got[:5]), 1.0)) < 1e-12
