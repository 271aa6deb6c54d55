"""A network packed on one stream and used on another: the use waits for the
packing launch, also when that stands behind other work.  Same statistics bit
for bit as packed and used on one stream."""
import pytest
import torch

import sde_mc_amd as sm
from sde_mc_amd import cv as CV
from sde_mc_amd import engine as E
from sde_mc_amd.nets import Mlp
from tests import jobs as J

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('layers', [[40], [50, 50, 50]])
def test_use_on_another_stream_waits_for_the_packing(layers):
    dev = E.require_device()
    torch.manual_seed(5)
    f, g = (Mlp(2, layers, 1, batch_norm=False, device=dev).eval() for _ in range(2))
    job = J.job_for(J.merton_sde(), 1.0, 40, 3000, grid='adapted', option=sm.EuroCall(1.0), seed=9)

    def run(nets):
        return CV.cv_simulate(job, *nets, int(job.max_steps), 0.02, 0.1, dev)[0]

    want = run([CV.DeviceNetwork(m, 2, 1, dev) for m in (f, g)]).clone()
    torch.cuda.synchronize()
    packing, using = torch.cuda.Stream(), torch.cuda.Stream()
    busy = torch.randn(4096, 4096, device=dev)
    # blocks of the words' sizes in the packing stream's pool hold other values
    with torch.cuda.stream(packing):
        stale = [torch.full((CV.BLOCK * CV.blocks(len(layers)),), 0x4100, dtype=torch.int16, device=dev)
                 for _ in range(4)]
        del stale
        for _ in range(20):
            busy = busy @ busy * 1e-3
        nets = [CV.DeviceNetwork(m, 2, 1, dev) for m in (f, g)]
    with torch.cuda.stream(using):
        got = run(nets)
    torch.cuda.synchronize()
    assert torch.equal(got, want)
