"""mc_simple asks a solver whose simulate_stats is not the library's for the
batches it was given, not for the merged launches of the fused estimator (no
GPU)."""
import pytest
import torch

import sde_mc_amd as sm
from tests import jobs as J


class _Recording(sm.JumpEulerSolver):
    def __init__(self, *args, **kw):
        super().__init__(*args, **kw)
        self.sizes = []

    def simulate_stats(self, n, option, discount, steps=None, coarse_factor=0):
        self.sizes.append(n)
        return float(n), float(2 * n), n


def _instance():
    solver = sm.JumpEulerSolver(J.merton_sde(), 1.0, 10, device='cpu', seed=1)
    solver.sizes = []

    def simulate_stats(n, *args, **kw):
        solver.sizes.append(n)
        return float(n), float(2 * n), n

    solver.simulate_stats = simulate_stats
    return solver


@pytest.mark.parametrize('make', [lambda: _Recording(J.merton_sde(), 1.0, 10, device='cpu', seed=1),
                                  _instance])
def test_own_simulate_stats_gets_its_batches(make):
    solver = make()
    st = sm.mc_simple(1000, solver, sm.EuroCall(1.0), sm.ConstantShortRate(0.02), bs=300)
    assert solver.sizes == [300, 300, 300, 100]
    assert st.sample_mean == 1.0
