"""A network packed on the device has the host packer's words exactly: every
depth, the narrowest and widest layers, batch norms on the inputs, after the
hidden layers and after the output, layers without bias; parameters the
packing kernel cannot read (fp64, on the host) go through the host."""
import pytest
import torch
import torch.nn as nn

from sde_mc_amd import cv as CV
from sde_mc_amd import engine as E
from sde_mc_amd.nets import Mlp

pytestmark = pytest.mark.gpu


def _randomise(net, seed):
    torch.manual_seed(seed)
    for m in net.modules():
        if isinstance(m, nn.BatchNorm1d):
            m.running_mean.normal_()
            m.running_var.uniform_(0.05, 3.0)
            if m.affine:
                nn.init.normal_(m.weight)
                nn.init.normal_(m.bias)
    return net.eval()


class _Seq(nn.Module):
    sequential = False

    def __init__(self, *mods):
        super().__init__()
        self.net = nn.Sequential(*mods)


def _cases():
    yield lambda: Mlp(2, [1], 1, batch_norm=False, batch_norm_init=False), 2, 1
    yield lambda: Mlp(2, [50, 50, 50], 1, batch_norm=False), 2, 1
    yield lambda: Mlp(5, [63, 63, 63, 63], 8), 5, 8
    yield lambda: Mlp(7, [33, 2], 3, batch_norm=True, batch_norm_init=False), 7, 3
    yield lambda: _Seq(nn.BatchNorm1d(3, affine=False), nn.Linear(3, 17, bias=False), nn.ReLU(),
                       nn.BatchNorm1d(17), nn.Linear(17, 5), nn.BatchNorm1d(5, eps=1e-2)), 3, 5
    yield lambda: _Seq(nn.Linear(2, 40), nn.BatchNorm1d(40), nn.BatchNorm1d(40), nn.ReLU(),
                       nn.Linear(40, 2)), 2, 2


@pytest.mark.parametrize('i', range(6))
@pytest.mark.parametrize('where', ['device', 'host', 'double'])
def test_device_words_equal_the_host_packers(i, where):
    make, n_in, n_out = list(_cases())[i]
    net = _randomise(make(), 40 + i)
    want, hidden = CV.pack_network(net, n_in, n_out)
    dev = E.require_device()
    if where == 'double':
        net = net.double()
    if where != 'host':
        net = net.to(dev)
    got = CV.DeviceNetwork(net, n_in, n_out, dev)
    entries, _ = CV._device_layers(CV.layer_plan(net), dev)
    assert (entries is not None) == (where == 'device' and i != 5)   # two norms in a row: the host
    assert got.hidden == hidden
    assert torch.equal(got.words.cpu(), torch.from_numpy(want.view('int16')))
