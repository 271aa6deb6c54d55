"""The Heston step of a fixed step size (carried root, reciprocal divisor) is
the general Euler step bit for bit: paths drawn in the kernel equal the
fixed-increment kernel's, which takes the general step, on the increments
they store.  Exact equality, no tolerance."""
import pytest
import torch

import sde_mc_amd as sm
from sde_mc_amd import _lib as L
from sde_mc_amd import engine as E
from tests import jobs as J

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('kappa,theta,xi,v0', [(0.25, 0.5, 0.3, 0.15),      # preset
                                               (1.5, 0.04, 0.3, 0.0),       # starts at zero
                                               (4.0, 0.01, 0.28, 1e-6),     # near the Feller bound
                                               (0.01, 90.0, 1.3, 25.0)])    # large variance
@pytest.mark.parametrize('steps,P', [(1, 1), (7, 65), (50, 1000), (400, 20000)])
def test_step_equals_the_general_step(kappa, theta, xi, v0, steps, P):
    dev = E.require_device()
    sde = sm.Heston(0.02, kappa, theta, xi, -0.6, torch.tensor([1.0, v0]))
    job = J.job_for(sde, 2.0, steps, P, option=sm.EuroCall(1.0), seed=77)
    paths = torch.empty((steps + 1, 2, P), dtype=torch.float32, device=dev)
    dw = torch.empty((steps, 2, P), dtype=torch.float32, device=dev)
    out = L.PathOut()
    out.paths_dev, out.normals_dev = paths.data_ptr(), dw.data_ptr()
    stored = E.simulate(job, dev, out=out)
    plain = E.simulate(job, dev)
    term = torch.empty((2, P), dtype=torch.float32, device=dev)
    fo = L.PathOut()
    fo.terminal_dev = term.data_ptr()
    fx = L.FixedIn()
    fx.dw_dev, fx.n_rows = dw.data_ptr(), steps
    fixed = E.simulate_fixed(job, fx, dev, out=fo)
    assert torch.isfinite(term).all()
    assert torch.equal(paths[-1], term)
    assert torch.equal(stored, fixed) and torch.equal(plain, fixed)
