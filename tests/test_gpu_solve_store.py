"""A stored solve writes every element it returns: poisoned memory shows up
nowhere, rows past a path's end hold its last state, zero increments and zero
marks, and the arrays agree with each other (exact)."""
import pytest
import torch

import sde_mc_amd as sm
from tests import jobs as J

pytestmark = pytest.mark.gpu


def _poison(n):
    """Fill the allocator's free memory with NaN, for the next torch.empty."""
    blocks = [torch.full((1 << 20,), float('nan'), device='cuda') for _ in range(n)]
    torch.cuda.synchronize()
    del blocks


@pytest.mark.parametrize('P', [1, 63, 64, 1000])
@pytest.mark.parametrize('model,steps', [('merton1', 1), ('merton1', 37), ('merton3', 12), ('levy2', 25)])
@pytest.mark.parametrize('grid', ['adapted', 'uniform'])
def test_jump_solver_arrays(model, steps, P, grid):
    _poison(24)
    sde = J.levy_rainbow_sde() if model == 'levy2' else J.merton_sde(rate=3.0, dim=int(model[-1]))
    s = sm.JumpEulerSolver(sde, 2.0, steps, device='cuda', seed=4, grid=grid)
    paths, (normals, times, left, total, jumps) = s.solve(P, return_normals=True)
    for t in (paths, normals, times, jumps) + (() if left is None else (left,)):
        assert torch.isfinite(t).all()
    assert paths.shape[1] == total + 1
    assert torch.all(jumps[:, 0] == 0)
    if grid == 'uniform':
        return
    t = times[:, :total + 1, 0]
    dt = torch.diff(t, dim=1)
    moving = dt > 0
    dw = normals[:, :total].reshape(P, total, -1)
    assert torch.all(dw[~moving] == 0) and torch.all(normals[:, total:] == 0)
    assert torch.all(paths[:, 1:][~moving] == paths[:, :-1][~moving])
    assert torch.all(left[:, 1:total + 1][~moving] == paths[:, 1:][~moving])
    jumped = (jumps[:, :total + 1] != 0).any(-1)
    assert torch.all(left[:, :total + 1][~jumped] == paths[~jumped])
    assert torch.all(jumps[:, total + 1:] == 0) and torch.all(left[:, total + 1:] == 0)
    assert torch.all(times[:, total + 1:] == 2.0)
    one = s.solve(0)
    assert one[0].shape[0] == 0


def test_diffusion_solver_arrays():
    _poison(24)
    for sde, cls in ((sm.Gbm(0.02, 0.3, torch.ones(3), 3), sm.EulerSolver),
                     (sm.DoubleGbm(0.02, 0.2, 0.1, torch.ones(2), 2), sm.EulerSolver),
                     (sm.Heston(0.02, 0.25, 0.5, 0.3, -0.3, torch.tensor([1.0, 0.15])), sm.HestonSolver)):
        paths, normals = cls(sde, 1.0, 21, device='cuda').solve(77, return_normals=True)
        assert torch.isfinite(paths).all() and torch.isfinite(normals).all()
