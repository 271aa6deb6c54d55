"""Batched launches with fewer, as many and more tiles than wavefronts, also
with more workgroups than the device holds at once: every tile runs once, so
the statistics equal the plain launches' bit for bit.  And a launch of few
tiles costs no more for the wavefronts that have none."""
import numpy as np
import pytest
import torch

import sde_mc_amd as sm
from sde_mc_amd import engine as E
from sde_mc_amd.batch import BatchRunner, BatchTune
from tests import jobs as J

pytestmark = pytest.mark.gpu

# one 64-path chunk of this many steps is a tile by itself
STEPS = {'merton': 120, 'levy': 60}


def _job(model, chunks, seed):
    sde = J.merton_sde() if model == 'merton' else J.levy_rainbow_sde(eps=0.4)
    return J.job_for(sde, 1.0, STEPS[model], max(1, 64 * chunks - 5), option=sm.EuroCall(1.0), seed=seed)


@pytest.mark.parametrize('wpb,bpc', [(1, 1), (4, 7), (8, 2), (2, 64)])
@pytest.mark.parametrize('model', ['merton', 'levy'])
@pytest.mark.parametrize('extra', [-1, 0, 1, 333])
def test_tiles_around_the_number_of_wavefronts(wpb, bpc, model, extra):
    dev = E.require_device()
    waves = torch.cuda.get_device_properties(dev).multi_processor_count * wpb * bpc
    total = waves + extra
    parts = [1, 2, max(1, total // 3)]
    parts.append(total - sum(parts))
    jobs = [_job(model, c, 50 + i) for i, c in enumerate(parts)]
    runner = BatchRunner(max_jobs=8, tune=BatchTune(waves_per_block=wpb, blocks_per_cu=bpc))
    got = runner.run(jobs)
    want = np.stack([E.simulate(j, dev).cpu().numpy() for j in jobs])
    assert np.array_equal(got, want)
    assert np.array_equal(runner.run(jobs), want)   # the counter starts anew


def _launch_us(tune, jobs, repeats=30):
    runner = BatchRunner(max_jobs=8, use_graph=False, tune=tune)
    best = 1e9
    ev = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
    for _ in range(repeats):
        runner.run(jobs, events=ev)
        best = min(best, 1e3 * ev[0].elapsed_time(ev[1]))
    return best


@pytest.mark.parametrize('model', ['merton', 'levy'])
def test_wavefronts_without_a_tile_cost_little(model):
    # 300 tiles in 1024 and in 7168 wavefronts (1.0; 2 to 3 when all took their first tile by atomics)
    jobs = [_job(model, 300, 7)]
    few = _launch_us(BatchTune(waves_per_block=4, blocks_per_cu=1), jobs)
    many = _launch_us(BatchTune(waves_per_block=4, blocks_per_cu=7), jobs)
    assert many < 1.5 * few
