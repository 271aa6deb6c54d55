"""Every element of every buffer a stored solve allocates is written: the
buffers themselves start as NaN (float32) or -1 (int32), whatever the allocator
held, and none of it is left, also in rows past every path's end."""
import pytest
import torch

import sde_mc_amd as sm
from tests import jobs as J
from tests.test_oracle_general import _general


def _unwritten(tensors):
    """Elements that still hold their buffer's poison."""
    return sum(int((torch.isnan(t) if t.is_floating_point() else t == -1).sum()) for t in tensors)


class _Poisoned:
    """torch.empty whose buffers start poisoned, and are kept."""

    def __init__(self, monkeypatch):
        self.kept = []
        empty = torch.empty

        def poisoned(*args, **kw):
            t = empty(*args, **kw)
            t.fill_(float('nan') if t.is_floating_point() else -1 if t.dtype == torch.int32 else 0)
            if t.dtype in (torch.float32, torch.int32):
                self.kept.append(t)
            return t

        monkeypatch.setattr(torch, 'empty', poisoned)


def test_the_check_finds_one_element():
    a, b = torch.zeros(3, 4), torch.zeros(5, dtype=torch.int32)
    assert _unwritten([a, b]) == 0
    a[2, 1] = float('nan')
    b[4] = -1
    assert _unwritten([a]) == 1 and _unwritten([a, b]) == 2


JUMPS = {
    'merton1': lambda: J.merton_sde(rate=3.0),
    'merton2': lambda: J.merton_sde(rate=3.0, dim=2),
    'merton3': lambda: J.merton_sde(rate=3.0, dim=3),
    'merton4': lambda: J.merton_sde(rate=3.0, dim=4),
    'no jumps': lambda: J.merton_sde(rate=0.0),
    'levy2 clock': lambda: J.levy_rainbow_sde(f=(0.2, 0.3), eps=0.4),
    'levy2 counts': lambda: J.levy_rainbow_sde(f=(0.2, 0.3)),
}


@pytest.mark.gpu
@pytest.mark.parametrize('P', [1, 63, 1000])
@pytest.mark.parametrize('steps', [1, 37])
@pytest.mark.parametrize('model', sorted(JUMPS))
@pytest.mark.parametrize('grid,low', [('adapted', False), ('adapted', True), ('uniform', False),
                                      ('uniform', True)])
def test_jump_solves(model, steps, P, grid, low, monkeypatch):
    s = sm.JumpEulerSolver(JUMPS[model](), 2.0, steps, device='cuda', seed=4, grid=grid)
    p = _Poisoned(monkeypatch)
    s.solve(P, return_normals=True, low_storage=low)
    assert len(p.kept) >= 1 and _unwritten(p.kept) == 0


DIFFUSIONS = {
    'gbm3': (lambda: sm.Gbm(0.02, 0.3, torch.ones(3), 3), 'EulerSolver'),
    'double2': (lambda: sm.DoubleGbm(0.02, 0.2, 0.1, torch.ones(2), 2), 'EulerSolver'),
    'heston': (lambda: sm.Heston(0.02, 0.25, 0.5, 0.3, -0.3, torch.tensor([1.0, 0.15])), 'HestonSolver'),
    'general 3 of 2': (lambda: _general(3, 2, seed=9), 'EulerSolver'),
    'general 1 of 1': (lambda: _general(1, 1, seed=9), 'EulerSolver'),
    'general 4 of 4': (lambda: _general(4, 4, seed=9), 'EulerSolver'),
}


@pytest.mark.gpu
@pytest.mark.parametrize('P', [1, 63, 1000])
@pytest.mark.parametrize('steps', [1, 37])
@pytest.mark.parametrize('model', sorted(DIFFUSIONS))
def test_diffusion_solves(model, steps, P, monkeypatch):
    make, solver = DIFFUSIONS[model]
    s = getattr(sm, solver)(make(), 1.0, steps, device='cuda', seed=4)
    p = _Poisoned(monkeypatch)
    s.solve(P, return_normals=True)
    assert len(p.kept) >= 2 and _unwritten(p.kept) == 0
