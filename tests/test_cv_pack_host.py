"""Which networks the packing kernel may read: parameters of host memory, and
vectors and matrices whose sizes do not belong together, go to the host packer,
which packs or refuses them as it always has (no GPU)."""
import numpy as np
import pytest
import torch

from sde_mc_amd import cv as CV
from sde_mc_amd.nets import Mlp


def test_host_parameters_are_packed_by_the_host():
    torch.manual_seed(1)
    m = Mlp(3, [20, 31], 2, batch_norm=False).eval()
    words, hidden = CV.pack_network(m, 3, 2)
    for device in (torch.device('cpu'), 'cpu'):
        net = CV.DeviceNetwork(m, 3, 2, device)
        assert net.hidden == hidden
        assert np.array_equal(net.words.numpy().view(np.uint16), words)


def _layers(model):
    return [m for m in model.modules() if isinstance(m, torch.nn.Linear)]


def _vector(n):
    return torch.nn.Parameter(torch.randn(n))


MISFITS = {
    'short batch norm on the inputs': lambda m: m.net.__setitem__(0, torch.nn.BatchNorm1d(1).eval()),
    'long batch norm on the inputs': lambda m: m.net.__setitem__(0, torch.nn.BatchNorm1d(9).eval()),
    'short batch norm after a layer': lambda m: m.net.__setitem__(2, torch.nn.BatchNorm1d(5).eval()),
    'short variance': lambda m: setattr(m.net[2], 'running_var', torch.rand(3)),
    'short bias': lambda m: setattr(_layers(m)[1], 'bias', _vector(4)),
    'weight of another width': lambda m: setattr(
        _layers(m)[1], 'weight', torch.nn.Parameter(torch.randn(31, 12))),
}


@pytest.mark.parametrize('misfit', sorted(MISFITS))
def test_misfitting_sizes_do_not_reach_the_packing_kernel(misfit):
    torch.manual_seed(2)
    m = Mlp(3, [20, 31], 2).eval()
    cpu = torch.device('cpu')
    assert CV._device_layers(CV.layer_plan(m), cpu)[0] is not None
    MISFITS[misfit](m)
    assert CV._device_layers(CV.layer_plan(m), cpu) == (None, None)


def test_replaced_weights_count_by_their_own_shape():
    torch.manual_seed(3)
    m = Mlp(3, [20, 31], 2, batch_norm=False).eval()
    first, second, _ = _layers(m)
    first.weight, first.bias = torch.nn.Parameter(torch.randn(24, 3)), _vector(24)
    second.weight = torch.nn.Parameter(torch.randn(31, 24))
    plan = CV.layer_plan(m)
    CV._check_shape(plan, 3, 2)
    entries, _ = CV._device_layers(plan, torch.device('cpu'))
    assert [(e.n_in, e.n_out) for e in entries] == [(3, 24), (24, 31), (31, 2)]
    words, _ = CV.pack_network(m, 3, 2)
    assert np.array_equal(CV.DeviceNetwork(m, 3, 2, 'cpu').words.numpy().view(np.uint16), words)
    first.weight = torch.nn.Parameter(torch.randn(70, 3))   # wider than the kernel's units
    with pytest.raises(NotImplementedError):
        CV._check_shape(CV.layer_plan(m), 3, 2)
