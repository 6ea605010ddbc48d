"""FP64 Gauss terms where a sum against the largest weight constant underflows:
zero weights (Student-t too), points of other modes, points far out.  Results against the
oracle (1e-12, the bar of the FP64 evals), and the kernel's time against that of
the same call on a plain sample: each pair is visited once wherever it lies."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _pair(oracle, kind, d, X, local_frac=0.2):
    import numcosmo_amd as na
    sd = (na.StatsDistVKDE if kind == 1 else na.StatsDistKDE).new(na.StatsDistKernelGauss.new(d))
    od = oracle.StatsDist(kind, 0, d, 0.0)
    for o in (sd, od):
        if kind == 1:
            o.set_local_frac(local_frac)
        o.add_obs_array(X)
        o.prepare()
    return sd, od


def _err(got, ref):
    return np.max(np.abs(got - ref) / np.maximum(np.abs(ref), 1.0))


@pytest.mark.parametrize("nu", [0.0, 3.0, 2.5])
@pytest.mark.parametrize("kind,d", [(0, 2), (1, 2), (1, 5), (1, 16), (0, 8)])
@pytest.mark.parametrize("m", [1, 70, 2100])
def test_zero_weights(kind, d, m, nu):
    """shrink = 0 leaves the zeros of the active set in the weights (the target is
    narrower than the sample, so that its outer kernels drop out; the sample is
    ordered outwards, so that whole splits have no weight)."""
    import numcosmo_amd as na
    g = np.random.default_rng(d)
    X = g.normal(size=(400, d))
    X = X[np.argsort(np.sum(X * X, 1))]
    k = na.StatsDistKernelGauss.new(d) if nu == 0.0 else na.StatsDistKernelST.new(d, nu)
    sd = (na.StatsDistVKDE if kind == 1 else na.StatsDistKDE).new(k)
    if kind == 1:
        sd.set_local_frac(0.2)
    sd.add_obs_array(X)
    sd.set_shrink(0.0)
    sd.prepare_interp(np.minimum(3.0 * np.sum(X * X, 1), 140.0))
    assert bool((sd.peek_weights() == 0.0).any())
    P = g.normal(size=(m, d))
    # the density from the device's own weights: two fits of a nearly singular
    # matrix differ in theirs
    w, href = sd.peek_weights(), sd.get_href()
    live = np.flatnonzero(w > 0.0)
    Ui = np.stack([np.linalg.inv(np.triu(sd.peek_cov_decomp(i))) for i in live])
    ln = np.array([sd.get_lnnorm(i) for i in live])
    Q = P[-20:]
    z = np.einsum("ikl,pik->pil", Ui, Q[:, None, :] - X[live]) / href
    chi2 = np.sum(z * z, 2)
    t = np.log(w[live]) - ln - (0.5 * chi2 if nu == 0.0 else 0.5 * (nu + d) * np.log1p(chi2 / nu))
    mx = t.max(1)
    ref = -2.0 * (mx + np.log(np.sum(np.exp(t - mx[:, None]), 1)))
    # 1e-11: the inverted factors' rounding times chi2
    assert _err(sd.eval_m2lnp_batch(P)[-20:], ref) < 1e-11


@pytest.mark.parametrize("kind,d", [(0, 4), (1, 4), (1, 12), (1, 13), (1, 16), (1, 36)])
@pytest.mark.parametrize("order", ["mixed", "sorted"])
@pytest.mark.parametrize("m", [1, 64, 500])
def test_separated_modes(oracle, kind, d, order, m):
    """Tight modes in every direction (so that the whitening does not bring them
    together), kernels shuffled and mode by mode, points in the modes and
    between them."""
    g = np.random.default_rng(d + m)
    k = d + 2
    n = k * (3 * d + 4)
    cen = g.uniform(-200.0, 200.0, size=(k, d))
    c = np.arange(n) % k
    c = np.sort(c) if order == "sorted" else c
    X = 0.3 * g.normal(size=(n, d)) + cen[c]
    sd, od = _pair(oracle, kind, d, X, local_frac=0.8 / k)
    P = 0.3 * g.normal(size=(m, d)) + cen[g.integers(0, k, size=m)] + 15.0 * (g.random(m) < 0.2)[:, None]
    assert _err(sd.eval_m2lnp_batch(P), od.eval_m2lnp_batch(P)) < 1e-12


@pytest.mark.parametrize("kind,d", [(0, 1), (1, 1), (0, 4), (1, 4), (1, 16), (1, 36)])
def test_outwards(oracle, kind, d):
    """Points from the centre to 1e5 widths out: sums against max b, between it
    and what underflows, and far below, in splits whose first kernel lies
    hundreds of powers of two under their nearest one."""
    g = np.random.default_rng(d)
    X = g.standard_t(4.0, size=(12 * d + 200, d))
    X[::7] *= 3.0
    sd, od = _pair(oracle, kind, d, X)
    u = g.normal(size=(400, d))
    P = u / np.linalg.norm(u, axis=1)[:, None] * np.exp(np.linspace(np.log(0.1), np.log(1e5), 400))[:, None]
    assert _err(sd.eval_m2lnp_batch(P), od.eval_m2lnp_batch(P)) < 1e-12
    assert _err(np.array([sd.eval_m2lnp(p) for p in P[::40]]), od.eval_m2lnp_batch(P[::40])) < 1e-12


@pytest.mark.parametrize("d,m", [(4, 20000), (16, 2048)])
def test_time_does_not_depend_on_the_weights_or_the_modes(d, m):
    """Each split once: 1.3 times the plain sample's kernel time at most.  The
    general form beside the fast one took 1.9 and 1.6 times at these sizes."""
    import torch

    import numcosmo_amd as na
    from numcosmo_amd._lib import check, lib
    g = np.random.default_rng(1)
    n = 4000
    Z, Zp = g.normal(size=(n, d)), g.normal(size=(m, d))
    k = d + 2
    cen = g.uniform(-200.0, 200.0, size=(k, d))
    far = cen[np.sort(g.integers(0, k, size=n))]
    farp = cen[g.integers(0, k, size=m)]

    def ms(X, P, m2lnp=None):
        sd = na.StatsDistVKDE.new(na.StatsDistKernelGauss.new(d))
        sd.set_local_frac(0.7 / k)
        sd.add_obs_array(X)
        if m2lnp is None:
            sd.prepare()
        else:
            sd.set_shrink(0.0)
            sd.prepare_interp(m2lnp)
            assert bool((sd.peek_weights() == 0.0).any())
        x = torch.tensor(P, device="cuda")
        out = torch.empty(m, dtype=torch.float64, device="cuda")
        check(lib().nckde_set_profiling(sd._h, 1))
        t = []
        for _ in range(12):
            check(lib().nckde_eval_m2lnp_device(sd._h, C.c_void_p(x.data_ptr()), m, C.c_void_p(out.data_ptr()), 0, None))
            f = C.c_float()
            check(lib().nckde_get_kernel_ms(sd._h, C.byref(f)))
            t.append(f.value)
        return np.median(t[2:])

    plain = ms(Z, Zp)
    zero = ms(Z, Zp, np.minimum(3.0 * np.sum(Z * Z, 1), 140.0))
    modes = ms(0.3 * Z + far, 0.3 * Zp + farp)
    print(f"d={d} m={m}: plain {1e3 * plain:.1f} us, zero weights {1e3 * zero:.1f}, modes {1e3 * modes:.1f}", flush=True)
    assert zero < 1.3 * plain
    assert modes < 1.3 * plain
