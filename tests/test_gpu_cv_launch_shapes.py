"""Control-variate launches around the size from which workgroups of eight
wavefronts are taken (2048 chunks of 64 paths) and the one up to which the 1-D
kernel holds the normals' products (3072), one and two networks, one and two
dimensions: every path's value is the one a small launch gives it, bit for
bit, and the last chunk's ragged end too."""
import pytest
import torch

import sde_mc_amd as sm
from sde_mc_amd import cv as CV
from sde_mc_amd import engine as E
from sde_mc_amd.nets import Mlp
from tests import jobs as J

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dim', [1, 2])
@pytest.mark.parametrize('nets', ['f', 'g', 'f and g'])
@pytest.mark.parametrize('chunks', [2047, 2048, 3072, 3073])
def test_values_do_not_depend_on_the_launch(dim, nets, chunks):
    dev = E.require_device()
    torch.manual_seed(dim)
    packed = [CV.DeviceNetwork(Mlp(dim + 1, [50, 50, 50], dim, batch_norm=False, device=dev).eval()
                               if which in nets.split() else None, dim + 1, dim, dev)
              for which in 'fg']
    sde, P = J.merton_sde(dim=dim), 64 * chunks - 3

    def gammas(first, n):
        job = J.job_for(sde, 1.0, 12, n, grid='adapted', option=sm.EuroCall(1.0), seed=3, path_offset=first)
        return CV.cv_simulate(job, *packed, int(job.max_steps), 0.02, 0.1, dev, gamma=True)[1]

    whole = gammas(0, P)
    for first in (0, 64 * 1000, 64 * 2046):
        n = min(64 * 9, P - first)
        assert torch.equal(whole[first:first + n], gammas(first, n))
