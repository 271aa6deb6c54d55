"""The adapted grid's row loop where it can go wrong: the step limit falling
inside and at the ends of a group of rows, few and many jumps per row, partial
wavefronts, stored and unstored paths.

Tolerance: the fp32 state against the fp64 oracle on the same Philox counters,
|x32 - x64| <= 2e-5 (1 + |x64|) as in the parity tests; step counts and the
limit are exact.
"""
import numpy as np
import pytest
import torch

import oracle
import sde_mc_amd as sm
from sde_mc_amd import _lib as L
from sde_mc_amd import engine as E
from tests import jobs as J

pytestmark = pytest.mark.gpu


def _run(job, store):
    dev = E.require_device()
    P, d = int(job.n_paths), job.model.dim
    term = torch.full((d, P), float('nan'), dtype=torch.float32, device=dev)
    ns = torch.full((P,), -1, dtype=torch.int32, device=dev)
    out = L.PathOut()
    out.terminal_dev, out.nsteps_dev = term.data_ptr(), ns.data_ptr()
    paths = None
    if store:
        paths = torch.empty((job.max_steps + 1, d, P), dtype=torch.float32, device=dev)
        out.paths_dev = paths.data_ptr()
    E.stats_to_host(E.simulate(job, dev, out=out))
    if store:
        assert torch.equal(paths[-1], term)   # rows past a path's end repeat its last state
    return term.cpu().numpy(), ns.cpu().numpy()


@pytest.mark.parametrize('rate', [0.0, 2.0, 60.0])
@pytest.mark.parametrize('model', ['merton1', 'merton4', 'levy2'])
@pytest.mark.parametrize('steps,P', [(1, 1), (5, 64), (6, 65), (13, 127)])
def test_rows_and_step_limit(model, rate, steps, P):
    if model == 'levy2':
        sde = J.levy_rainbow_sde(eps=0.05 if rate else 0.5)
    else:
        sde = J.merton_sde(rate=rate, dim=int(model[-1]))
    job = J.job_for(sde, 1.5, steps, P, grid='adapted', seed=900 + steps, option=sm.EuroCall(1.0))
    _, want, ns = oracle.simulate(job, 0, P)
    for store in (False, True):
        term, got = _run(job, store)
        assert np.array_equal(got, ns)
        assert np.all(np.abs(term - want[0]) <= 2e-5 * (1 + np.abs(want[0])))
    # the limit: the longest path's own length is enough, one step less is not
    job.max_steps = int(ns.max())
    term, got = _run(job, False)
    assert np.array_equal(got, ns)
    if job.max_steps > 1:
        job.max_steps -= 1
        with pytest.raises(L.SdemcError, match='max_steps'):
            _run(job, False)
