"""The uniform grid's step loop compiled for a family's common form against the
general loop (which storing kernels run): the same sums bit for bit, at step
counts around the loop's strides (4 and 6 steps, two groups a turn, windows of
8), without jumps, with few, and with more than a jump queue holds; jobs whose
coefficients have no common form; single launches and the batched kernels;
coupled pairs against the oracle (2e-5 (1 + |x|), the parity tolerance)."""
import numpy as np
import pytest
import torch

import oracle
import sde_mc_amd as sm
from sde_mc_amd import _lib as L
from sde_mc_amd import engine as E
from sde_mc_amd.batch import BatchRunner
from tests import jobs as J

pytestmark = pytest.mark.gpu

MODELS = {
    'gbm1': lambda: J.merton_sde(rate=0.0),
    'merton1': lambda: J.merton_sde(rate=2.0),
    'merton1_dense': lambda: J.merton_sde(rate=80.0),
    'merton3': lambda: J.merton_sde(rate=5.0, dim=3),
    'loggbm': lambda: sm.LogGbm(0.02, 0.2, torch.tensor([0.0])),
    'levy2_counts': lambda: J.levy_rainbow_sde(f=(0.2, 0.3)),
    'levy2_clock': lambda: J.levy_rainbow_sde(f=(0.2, 0.3), eps=0.4),
    'levy2_linear': lambda: sm.LevyRainbow.default_params(4, 'cpu').solver.sde,
}


def _job(model, N, P, coupled=0, exact=False):
    return J.job_for(MODELS[model](), 1.0, N, P, coarse_factor=coupled, exact_jumps=exact,
                     option=sm.EuroCall(0.9), seed=100 + N)


@pytest.mark.parametrize('model', sorted(MODELS))
@pytest.mark.parametrize('N', [1, 3, 4, 5, 6, 7, 8, 9, 11, 12, 13, 17, 24, 25, 53])
def test_common_form_equals_the_general_loop(model, N):
    dev = E.require_device()
    P = 193
    jobs = [_job(model, N, P), _job(model, N, P, exact=True)]
    plain = [E.simulate(j, dev) for j in jobs]
    for j, want in zip(jobs, plain):
        paths = torch.empty((N + 1, j.model.dim, P), dtype=torch.float32, device=dev)
        out = L.PathOut()
        out.paths_dev = paths.data_ptr()
        assert torch.equal(E.simulate(j, dev, out=out), want)
    got = BatchRunner(max_jobs=8).run(jobs)
    assert np.array_equal(got, np.stack([p.cpu().numpy() for p in plain]))


@pytest.mark.parametrize('model', ['gbm1', 'merton1', 'merton1_dense', 'levy2_counts', 'levy2_clock'])
@pytest.mark.parametrize('N,M', [(2, 2), (6, 3), (12, 2), (28, 4)])
def test_coupled_pairs_against_the_oracle(model, N, M):
    dev = E.require_device()
    P = 130
    job = _job(model, N, P, coupled=M)
    term = torch.empty((2, job.model.dim, P), dtype=torch.float32, device=dev)
    out = L.PathOut()
    out.terminal_dev = term.data_ptr()
    E.stats_to_host(E.simulate(job, dev, out=out))
    _, want, _ = oracle.simulate(job, 0, P)
    assert np.all(np.abs(term.cpu().numpy() - want) <= 2e-5 * (1 + np.abs(want)))
