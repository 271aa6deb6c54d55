"""Parameter gradients of a tall Linear layer against fp64, at the edges of the
tiles (1, 31, 32, 33, 63, 64 columns), of a row pair, a wavefront's rows and
the workgroup count.

Tolerance: each result is a sum of products, every product exact inside its
fused multiply-add; one rounding per row of a wavefront (at most 128 here),
per wavefront of a workgroup (4), per partial of a sixteenth of the
workgroups (16) and per sixteenth (16), so |error| <= 164 2^-24 sum |x dy|.
"""
import pytest
import torch

import sde_mc_amd as sm
from sde_mc_amd import _lib as L
from sde_mc_amd import engine as E
from sde_mc_amd import varred as V

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('rows', [1, 2, 63, 64, 257, 4096, 65537, 100003])
@pytest.mark.parametrize('n_in,n_out', [(1, 1), (2, 50), (31, 32), (32, 33), (50, 50), (50, 1),
                                        (63, 64)])
def test_gradients_against_fp64(rows, n_in, n_out):
    torch.manual_seed(rows + n_in)
    x = torch.randn(rows, n_in, device='cuda')
    dy = torch.randn(rows, n_out, device='cuda')
    dw, db = E.linear_grads(x, dy)
    X, Y = x.double().cpu(), dy.double().cpu()
    eps = 164 * 2.0 ** -24
    assert torch.all((dw.double().cpu() - Y.t() @ X).abs() <= eps * (Y.abs().t() @ X.abs()))
    assert torch.all((db.double().cpu() - Y.sum(0)).abs() <= eps * Y.abs().sum(0))


def test_non_finite_values_reach_only_their_products():
    x, dy = torch.ones(3000, 3, device='cuda'), torch.ones(3000, 2, device='cuda')
    x[7, 1], dy[2999, 0] = float('inf'), float('nan')
    dw, db = E.linear_grads(x, dy)
    assert torch.isnan(dw[0]).all() and torch.isnan(db[0])
    assert dw[1].tolist() == [3000.0, float('inf'), 3000.0] and db[1] == 3000.0


def test_sizes_outside_the_kernel_are_refused():
    x = torch.zeros(8, 64, device='cuda')
    with pytest.raises(L.SdemcError):
        E.linear_grads(x, torch.zeros(8, 2, device='cuda'))
    with pytest.raises(L.SdemcError):
        E.linear_grads(x[:, :2].contiguous(), torch.zeros(8, 65, device='cuda'))


def test_the_training_forward_is_the_modules():
    torch.manual_seed(1)
    net = sm.Mlp(3, [63, 20], 2, device='cuda')
    x = torch.randn(V.MIN_SPLIT_POINTS, 3, device='cuda')
    f = V._training_forward(net)
    assert f is not net and f.sequential is False
    want = net(x)
    assert torch.equal(f(x), want) and torch.equal(f(x[:5]), net(x[:5]))
    for name, hook in (('forward', lambda m, i, o: None), ('forward_pre', lambda m, i: None)):
        h = getattr(net.net[1], 'register_%s_hook' % name)(hook)
        assert V._training_forward(net) is net
        h.remove()
    assert V._training_forward(sm.Lstm(3, 4, 1, device='cuda')).sequential
