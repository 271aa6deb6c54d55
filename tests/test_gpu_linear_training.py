"""The training forward's gradients against fp64: one Linear layer (dx, dw, db,
a missing bias, frozen parameters, an expanded dy), whole networks, and second
derivatives, which the split kernel does not carry itself.

Bounds, u = 2^-24: an fp32 dot product of n terms, in any order, is off by at
most n u sum |terms| to first order.  Through a network every value carries the
relative errors of the products before it, so a gradient of depth L over `rows`
points is held to (rows + 2 L (width + 2)) u times the same chain of absolute
values."""
import pytest
import torch

from sde_mc_amd import engine as E
from sde_mc_amd import varred as V
from sde_mc_amd.nets import Mlp

pytestmark = pytest.mark.gpu
U = 2.0 ** -24
ROWS = V.MIN_SPLIT_POINTS + 77


def _net(layers, out=1, bias=True, seed=1):
    torch.manual_seed(seed)
    dev = E.require_device()
    m = Mlp(3, layers, out, batch_norm=False, batch_norm_init=False, device=dev)
    if not bias:
        for lin in _linears(m):
            lin.bias = None
    return m


def _linears(m):
    return [q for q in m.net if isinstance(q, torch.nn.Linear)]


@pytest.mark.parametrize('n_in,n_out', [(1, 1), (31, 33), (63, 64), (50, 50)])
@pytest.mark.parametrize('what', ['all', 'no bias', 'frozen weight', 'frozen bias', 'weight alone',
                                  'expanded dy'])
def test_one_layer(n_in, n_out, what):
    dev = E.require_device()
    torch.manual_seed(n_in)
    x = torch.randn(ROWS, n_in, device=dev, requires_grad=what != 'weight alone')
    w = torch.randn(n_out, n_in, device=dev, requires_grad=what != 'frozen weight')
    b = None if what == 'no bias' else torch.randn(n_out, device=dev,
                                                   requires_grad=what != 'frozen bias')
    y = V._Linear.apply(x, w, b)
    if what == 'expanded dy':
        dy = torch.ones((), device=dev).expand(ROWS, n_out)
        y.sum().backward()
    else:
        dy = torch.randn(n_out, ROWS, device=dev).t()
        y.backward(dy)
    X, W, D = x.detach().double(), w.detach().double(), dy.double()
    for t, value, size in ((x, D @ W, n_out * (D.abs() @ W.abs())),
                           (w, D.t() @ X, ROWS * (D.abs().t() @ X.abs())),
                           (b, D.sum(0), ROWS * D.abs().sum(0))):
        if t is None or not t.requires_grad:
            assert t is None or t.grad is None
            continue
        assert ((t.grad.double() - value).abs() <= U * size).all()


@pytest.mark.parametrize('layers', [[50], [50, 50, 50], [7, 63, 20]])
@pytest.mark.parametrize('bias', [True, False])
def test_whole_network(layers, bias):
    m = _net(layers, bias=bias)
    frozen = _linears(m)[1].weight
    frozen.requires_grad_(False)
    forward = V._training_forward(m)
    assert forward is not m
    x = torch.randn(ROWS, 3, device=E.require_device(), requires_grad=True)
    dy = torch.randn(ROWS, 1, device=x.device)
    forward(x).backward(dy)
    # the same chain in fp64, and its absolute values
    lins = _linears(m)
    a, size = [x.detach().double()], [x.detach().double().abs()]
    masks = []
    for q, lin in enumerate(lins):
        W = lin.weight.detach().double()
        c = lin.bias.detach().double() if bias else W.new_zeros(W.shape[0])
        z, s = a[-1] @ W.t() + c, size[-1] @ W.abs().t() + c.abs()
        if q + 1 < len(lins):
            masks.append(z > 0)
            # units too near zero for the fp32 sign to be certain
            assert ((z.abs() > 200 * U * s) | (z == 0)).double().mean() > 0.99
            z = z.clamp(min=0)
        a.append(z)
        size.append(s)
    d, ds = dy.double(), dy.double().abs()
    width, n = max(layers), ROWS
    factor = (n + 2 * len(lins) * (width + 2)) * U
    for q in reversed(range(len(lins))):
        lin = lins[q]
        W = lin.weight.detach().double()
        if lin.weight is frozen:
            assert lin.weight.grad is None
        else:
            bound = factor * (ds.t() @ size[q])
            assert ((lin.weight.grad.double() - d.t() @ a[q]).abs() <= bound).all()
        if bias:
            assert ((lin.bias.grad.double() - d.sum(0)).abs() <= factor * ds.sum(0)).all()
        d, ds = d @ W, ds @ W.abs()
        if q:
            d, ds = d * masks[q - 1], ds
    assert ((x.grad.double() - d).abs() <= factor * ds).all()


@pytest.mark.parametrize('bias', [True, False])
def test_second_derivatives_are_the_modules(bias):
    m = _net([20, 30], bias=bias)
    forward = V._training_forward(m)
    x = torch.randn(ROWS, 3, device=E.require_device())
    out = []
    for call in (forward, m):
        params = list(m.parameters())
        first = torch.autograd.grad(call(x).square().mean(), params, create_graph=True)
        total = sum((g * g).sum() for g in first)
        out.append(torch.autograd.grad(total, params))
    for g, want in zip(*out):
        scale = want.abs().max().item()
        assert scale > 0
        assert (g - want).abs().max().item() <= 1e-4 * scale
