"""Batched and plain jobs and the step form of their coefficients: a uniform-grid
job takes its family's common step or the general one, in kernels of their own
(plain, generic class) or side by side (dedicated classes), single-level or
coupled; a job's statistics are the same bits either way (same chunks, same
sums)."""
import pytest
import torch

import sde_mc_amd as sm
from sde_mc_amd import engine as E
from tests import jobs as J


def _job(dim, coarse, mixed, n_paths=200, steps=27, rate=3.0, law='normal'):
    if law == 'levy':
        sde = J.levy_rainbow_sde(f=(0.2, 0.2))
    else:
        sde = J.merton_sde(rate=rate, dim=dim)
    job = J.job_for(sde, 0.75, steps, n_paths, option=sm.EuroCall(1.0),
                    coarse_factor=3 if coarse else 0)
    if mixed:  # neither constant nor proportional
        for i in range(job.model.dim):
            job.model.b0[i], job.model.b1[i] = 0.05, 0.15
    return job


CASES = [(dim, law, coarse) for dim, law in ((1, 'normal'), (2, 'levy'), (3, 'normal'))
         for coarse in (False, True)]


@pytest.mark.gpu
@pytest.mark.parametrize('n_paths,steps', [(1, 1), (63, 3), (130, 4), (1000, 27)])
def test_batched_equals_plain(n_paths, steps):
    from sde_mc_amd.batch import BatchRunner, chunks_of
    dev = E.require_device()
    jobs = [_job(dim, coarse and steps % 3 == 0, mixed, n_paths, steps, law=law)
            for dim, law, coarse in CASES for mixed in (False, True)]
    runner = BatchRunner(max_jobs=len(jobs), partial_chunks=sum(chunks_of(j.n_paths) for j in jobs))
    rows = runner.run(jobs)
    for row, job in zip(rows, jobs):
        s = E.simulate(job, dev)
        assert [float(v) for v in row[:2]] == [float(s[0]), float(s[1])]
