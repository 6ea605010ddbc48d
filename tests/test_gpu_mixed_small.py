"""Mixed evals on both sides of the lines below which the FP64 form runs instead:
which form ran (the FP64 one gives the FP64 eval's results to the bit, the
mixed one never does on these samples), and its error against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _pair(oracle, kind, nu, d, n):
    import numcosmo_amd as na
    g = np.random.default_rng(100 * d + n)
    X = g.normal(size=(n, d))
    k = na.StatsDistKernelGauss.new(d) if nu == 0.0 else na.StatsDistKernelST.new(d, nu)
    sd = (na.StatsDistVKDE if kind == 1 else na.StatsDistKDE).new(k)
    od = oracle.StatsDist(kind, 0 if nu == 0.0 else 1, d, nu)
    for o in (sd, od):
        if kind == 1:
            o.set_local_frac(max(0.05, (2.0 * d + 20.0) / n))
        o.add_obs_array(X)
        o.prepare()
    # a sample whose probe would send the handle to FP64 stays on the mixed
    # form; its error is held to ten times the probe's instead of 1e-6
    sd.set_mixed_tolerance(1e-3)
    err, fallback = sd.get_mixed_check()
    assert not fallback
    return sd, od, g, max(1e-6, 10.0 * err)


# kind, nu, d, n, m of the last FP64 call, m of the first mixed one
LINES = [
    (1, 3.0, 3, 12001, 64, 65),
    (1, 3.0, 3, 2501, 299, 300),
    (1, 2.5, 7, 7501, 64, 65),
    (1, 2.5, 7, 2001, 239, 240),
    (1, 3.0, 8, 6001, 128, 129),
    (1, 2.5, 12, 5003, 128, 129),
    (1, 2.5, 12, 2001, 299, 300),
    (1, 3.0, 16, 4001, 256, 257),
    (1, 0.0, 16, 5001, 192, 193),
    (1, 2.5, 15, 4501, 128, 129),
    (1, 3.0, 24, 701, 713, 714),
    (1, 0.0, 32, 3001, 256, 257),
    (1, 3.0, 40, 3001, 256, 257),
    (1, 0.0, 41, 8001, 128, 129),
    (1, 3.0, 49, 8001, 128, 129),
    (1, 3.0, 64, 3001, 256, 257),
    (1, 0.0, 60, 8001, 128, 129),
    (1, 2.5, 64, 4001, 187, 188),
    (0, 3.0, 8, 6001, 128, 129),
    (0, 0.0, 16, 3001, 256, 257),
    (1, 3.0, 8, 301, 2048, 2049),
]


@pytest.mark.parametrize("kind,nu,d,n,below,above", LINES)
def test_both_sides_of_the_lines(oracle, kind, nu, d, n, below, above):
    sd, od, g, bar = _pair(oracle, kind, nu, d, n)
    P = g.normal(size=(above, d))
    few = sd.eval_m2lnp_batch(P[:below], 1)
    assert np.array_equal(few, sd.eval_m2lnp_batch(P[:below], 0))
    got = sd.eval_m2lnp_batch(P, 1)
    assert not np.array_equal(got, sd.eval_m2lnp_batch(P, 0))
    ref = od.eval_m2lnp_batch(P)
    rel = np.maximum(np.abs(ref), 1.0)
    assert np.max(np.abs(few - ref[:below]) / rel[:below]) < 1e-12
    assert np.max(np.abs(got - ref) / rel) < bar
