"""The bias gradient of the split kernel is as precise as fp32 holds it: column
sums in fp64, rounded once.

Bound: 2^-24 |sum| of the last rounding; in fp64 at most 64 rows of a lane, 8
lanes, 16 workgroups and 16 sixteenths one after another (for up to 131072 rows),
104 2^-53 sum |dy|; a workgroup's sum kept as two floats, 2^-48 of it.  (As a column
of the fp32 product it was off by up to 1.8 times what torch's sum is.)"""
import pytest
import torch

from sde_mc_amd import engine as E

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('rows', [1, 65, 2048, 8000, 50000, 100003])
@pytest.mark.parametrize('n_in,n_out', [(2, 1), (32, 33), (52, 52), (63, 64)])
@pytest.mark.parametrize('mean', [0.0, 1.0])
def test_column_sums(rows, n_in, n_out, mean):
    torch.manual_seed(rows)
    x = torch.randn(rows, n_in, device='cuda')
    dy = torch.randn(rows, n_out, device='cuda') * 1e-3 + mean
    _, db = E.linear_grads(x, dy)
    want, size = dy.double().sum(0), dy.double().abs().sum(0)
    bound = 2.0 ** -24 * want.abs() * (1 + 2.0 ** -20) + (104 * 2.0 ** -53 + 2.0 ** -47) * size
    assert ((db.double() - want).abs() <= bound).all()


def test_infinities_and_nan():
    dy = torch.ones(5000, 4, device='cuda')
    dy[4999, 0], dy[0, 1], dy[7, 2] = float('inf'), -float('inf'), float('nan')
    _, db = E.linear_grads(torch.ones(5000, 2, device='cuda'), dy)
    assert db[0] == float('inf') and db[1] == -float('inf') and torch.isnan(db[2]) and db[3] == 5000
