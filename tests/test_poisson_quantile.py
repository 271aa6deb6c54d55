"""The Poisson quantile behind the jump caps: scipy.stats' value over the rates a
job may have (the caps size buffers, so they must not move by one), and the
defining property where the distribution function is well away from 1."""
import numpy as np
import pytest
from scipy.stats import poisson

from sde_mc_amd import engine as E


@pytest.mark.parametrize('q', [0.5, 1 - 1 / 1e9, 1 - 1e-15])
def test_equals_scipy(q):
    rng = np.random.default_rng(3)
    mus = np.concatenate([10 ** rng.uniform(-8, 5, 4000), np.arange(1, 1200) * 0.25])
    got = np.array([E.poisson_quantile(q, float(m)) for m in mus])
    assert np.array_equal(got, poisson.ppf(q, mus))


def test_is_the_quantile():
    for mu in (0.01, 0.7, 6.0, 123.5, 2000.0):
        k = E.poisson_quantile(0.999, mu)
        assert poisson.cdf(k, mu) >= 0.999 and (k == 0 or poisson.cdf(k - 1, mu) < 0.999)
