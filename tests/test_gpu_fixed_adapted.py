"""Jump-adapted paths from caller-supplied inputs against the oracle: one to
four components, both jump updates, jumps at the same time, at a grid time, at
the horizon and a step limit that ends paths.  2e-5 (1 + |x|), the parity
tolerance; step counts exact."""
import numpy as np
import pytest

import oracle
import sde_mc_amd as sm
from sde_mc_amd import _lib as L
from tests import jobs as J
from tests.test_gpu_parity import TOL, _close, _run_fixed

pytestmark = pytest.mark.gpu


def _job(model, dim, exact):
    sde = J.merton_sde(rate=5.0, dim=dim) if model == 'merton' else J.levy_rainbow_sde(eps=0.4)
    return J.job_for(sde, 1.0, 16, 777, grid='adapted', option=sm.EuroCall(1.0), exact_jumps=exact)


@pytest.mark.parametrize('model,dim', [('merton', 1), ('merton', 2), ('merton', 3), ('merton', 4),
                                       ('levy', 2)])
@pytest.mark.parametrize('exact', [False, True])
def test_ties_and_edges(model, dim, exact):
    job = _job(model, dim, exact)
    fx = J.fixed_adapted(job, seed=21)
    jt = fx.a['jt']
    jt[1, ::3] = jt[0, ::3]                      # two jumps at once
    jt[0, 1::3] = np.float32(4 / 16)             # at a grid time
    jt[0, 2::3] = np.float32(1.0)                # at the horizon
    jt[:] = np.sort(jt, axis=0)
    _, term, ns, _ = _run_fixed(job, fx)
    _, oterm, ons = oracle.simulate_fixed(job, fx.host_struct(), int(job.n_paths))
    assert _close(term, oterm) < TOL
    assert np.array_equal(ns, ons)


def test_a_path_past_the_step_limit_is_reported():
    job = _job('merton', 1, False)
    fx = J.fixed_adapted(job, seed=22)
    job.max_steps = 17
    *_, stats = _run_fixed(job, fx)   # the raw statistics, unchecked
    assert int(stats[3]) & L.FLAG_OVERFLOW
