"""Which models the training loops call through their own forward: anything
but a plain Mlp of a plain Sequential keeps the module's call (no GPU)."""
import torch

from sde_mc_amd import varred as V
from sde_mc_amd.nets import Mlp


class _Wrapped(torch.nn.Module):
    """A network put in place of Mlp.net that cannot be iterated."""

    def __init__(self, inner):
        super().__init__()
        self.inner = inner

    def forward(self, x):
        return self.inner(x)


def test_a_replaced_net_keeps_the_modules_call():
    m = Mlp(2, [5], 1, batch_norm=False)
    m.net = _Wrapped(m.net)
    assert V._training_forward(m) is m
    m.net = torch.nn.Linear(2, 1)
    assert V._training_forward(m) is m
