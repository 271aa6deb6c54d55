"""Batches of a dataset whose arrays lie on several devices equal the ones
stacked from single trajectories, each on its own device (exact)."""
import pytest
import torch
from torch.utils.data import DataLoader

from sde_mc_amd.nets import NormalPathData, PathLoader

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('devices', [('cuda', 'cpu', 'cuda'), ('cpu', 'cuda', 'cuda'), ('cpu', 'cpu', 'cuda')])
def test_arrays_on_several_devices(devices):
    torch.manual_seed(6)
    paths, pay, normals = (t.to(d) for t, d in zip(
        (torch.randn(31, 5, 2), torch.randn(31), torch.randn(31, 4, 2)), devices))
    ds = NormalPathData(paths, pay, normals)
    for (got, gp), (want, wp) in zip(PathLoader(ds, batch_size=8), DataLoader(ds, batch_size=8)):
        for g, w in zip(list(got) + [gp], list(want) + [wp]):
            assert g.device == w.device and torch.equal(g, w)
