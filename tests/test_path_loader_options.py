"""A PathLoader with options of its own, and its place in the random stream,
against the DataLoader it stands for (no GPU)."""
import pytest
import torch
from torch.utils.data import DataLoader

from sde_mc_amd.nets import NormalPathData, PathLoader


def _data(n=23):
    g = torch.Generator().manual_seed(4)
    return NormalPathData(torch.randn(n, 6, 2, generator=g), torch.randn(n, generator=g),
                          torch.randn(n, 5, 2, generator=g))


def _marked(rows):
    return [r[1] for r in rows], 'mark'


@pytest.mark.parametrize('set_later', [False, True])
def test_own_collate_function_is_used(set_later):
    ds = _data()
    if set_later:
        dl = PathLoader(ds, batch_size=5)
        dl.collate_fn = _marked
    else:
        dl = PathLoader(ds, batch_size=5, collate_fn=_marked)
    assert all(batch[1] == 'mark' for batch in dl)


def test_without_batches():
    ds = _data()
    got = list(PathLoader(ds, batch_size=None))
    assert len(got) == len(ds) and torch.equal(got[3][1], ds[3][1])


def test_workers_are_used():
    seen = []
    dl = PathLoader(_data(), batch_size=6, num_workers=1, worker_init_fn=seen.append)
    it = iter(dl)
    assert type(it).__module__.startswith('torch.utils.data')
    del it


@pytest.mark.parametrize('generator', [False, True])
def test_seed_between_the_iteration_and_its_first_batch(generator):
    ds = _data()
    order = []
    for cls in (DataLoader, PathLoader):
        g = torch.Generator().manual_seed(8) if generator else None
        torch.manual_seed(1)
        it = iter(cls(ds, batch_size=4, shuffle=True, generator=g))
        torch.manual_seed(2)
        order.append([payoffs for _, payoffs in it] + [torch.rand(2)])
    assert all(torch.equal(a, b) for a, b in zip(*order))
