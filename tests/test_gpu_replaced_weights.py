"""Linear layers whose weights were replaced by ones of another size train by
the weights' own shape: wider than the split kernel takes, they keep the
module's call."""
import pytest
import torch

from sde_mc_amd import engine as E
from sde_mc_amd import varred as V
from sde_mc_amd.nets import Mlp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('width', [40, 64, 90])
def test_replaced_weights_train(width):
    dev = E.require_device()
    torch.manual_seed(3)
    m = Mlp(2, [20, 20], 1, batch_norm=False, batch_norm_init=False, device=dev)
    first, second, _ = [q for q in m.net if isinstance(q, torch.nn.Linear)]
    first.weight = torch.nn.Parameter(torch.randn(width, 2, device=dev))
    first.bias = torch.nn.Parameter(torch.randn(width, device=dev))
    second.weight = torch.nn.Parameter(torch.randn(20, width, device=dev))
    x = torch.randn(V.MIN_SPLIT_POINTS, 2, device=dev)
    grads = []
    for call in (V._training_forward(m), m):
        m.zero_grad()
        call(x).square().sum().backward()
        grads.append([p.grad.clone() for p in m.parameters()])
    for g, want in zip(*grads):
        assert (g - want).abs().max() <= 1e-3 * want.abs().max()
