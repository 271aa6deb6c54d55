"""The carried root of the Heston step is sqrt(v) also where the implicit root
vanishes: almost on the Feller bound and from v = 0 the constant term is lost
beside B^2, and the hardware root may leave the quotient one unit below zero.
Paths drawn in the kernel equal, bit for bit, the fixed-increment kernel's on
the increments they store; it takes the root of the stored v, never negative."""
import pytest
import torch

import sde_mc_amd as sm
from sde_mc_amd import _lib as L
from sde_mc_amd import engine as E
from tests import jobs as J

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('kappa,xi', [(1.0, 3.0), (0.3, 7.0), (0.01, 1.7), (2.0, 0.9), (0.05, 20.0)])
@pytest.mark.parametrize('steps,T', [(8, 8.0), (40, 20.0), (200, 1.0)])
@pytest.mark.parametrize('coupled', [0, 2])
def test_step_equals_the_general_step_on_the_feller_bound(kappa, xi, steps, T, coupled):
    dev = E.require_device()
    P = 50000
    theta = xi * xi * (1 + 1e-7) / (2 * kappa)
    sde = sm.Heston(0.02, kappa, theta, xi, -0.6, torch.tensor([1.0, 0.0]))
    job = J.job_for(sde, T, steps, P, option=sm.EuroCall(1.0), seed=77)
    dw = torch.empty((steps, 2, P), dtype=torch.float32, device=dev)
    out = L.PathOut()
    out.normals_dev = dw.data_ptr()
    paths = torch.empty((steps + 1, 2, P), dtype=torch.float32, device=dev)
    out.paths_dev = paths.data_ptr()
    E.simulate(job, dev, out=out)
    job = J.job_for(sde, T, steps, P, coarse_factor=coupled, option=sm.EuroCall(1.0), seed=77)
    lv = 2 if coupled else 1
    drawn, given = (torch.empty((lv, 2, P), dtype=torch.float32, device=dev) for _ in range(2))
    for term, run in ((drawn, lambda o: E.simulate(job, dev, out=o)),
                      (given, lambda o: E.simulate_fixed(job, fx, dev, out=o))):
        fx = L.FixedIn()
        fx.dw_dev, fx.n_rows = dw.data_ptr(), steps
        o = L.PathOut()
        o.terminal_dev = term.data_ptr()
        run(o)
    assert torch.equal(drawn.view(torch.int32), given.view(torch.int32))
