"""Which networks the packing kernel may read: parameters of host memory, and
vectors and matrices whose sizes do not belong together, go to the host packer,
which packs or refuses them as it always has (no GPU)."""
import numpy as np
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
