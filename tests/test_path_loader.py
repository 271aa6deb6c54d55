"""Batches gathered array by array equal the ones stacked from single
trajectories, in the same order for the same seed (exact): on the CPU through
torch, on the device through the gather kernel, for the layouts the solvers
store (path index fastest) and others, odd sizes and the last ragged batch."""
import pytest
import torch
from torch.utils.data import DataLoader

from sde_mc_amd import engine as E
from sde_mc_amd.nets import AdaptedPathData, NormalPathData, PathLoader


def _stored(P, rows, dim, dev, tail=()):
    """(P, rows, dim) view of [rows][dim][P] storage."""
    t = torch.randn((rows, dim) + tail + (P,))
    return t.permute(*([t.dim() - 1] + list(range(t.dim() - 1)))).to(dev)


def _datasets(P, rows, dim, dev):
    torch.manual_seed(P + rows)
    pay = torch.randn(P).to(dev)
    yield NormalPathData(_stored(P, rows + 1, dim, dev), pay, _stored(P, rows, dim, dev))
    yield NormalPathData(_stored(P, rows + 1, dim, dev), pay, _stored(P, rows, dim, dev, (2,)))
    yield AdaptedPathData(_stored(P, rows + 1, dim, dev), pay, _stored(P, rows, dim, dev),
                          _stored(P, rows + 1, dim, dev), _stored(P, rows + 1, 1, dev),
                          _stored(P, rows + 1, dim, dev)[:, :, :], rows)
    # storage the kernel's two strides cannot describe, and contiguous rows
    odd = torch.randn(P, rows + 1, 2 * dim, 2)[:, :, ::2].to(dev)
    yield NormalPathData(odd, pay, torch.randn(P, rows, dim).to(dev))


@pytest.mark.parametrize('dev', ['cpu', pytest.param('cuda', marks=pytest.mark.gpu)])
@pytest.mark.parametrize('P,rows,dim,bs', [(1, 1, 1, 1), (37, 5, 2, 8), (257, 33, 4, 100)])
@pytest.mark.parametrize('shuffle', [False, True])
def test_gathered_batches_equal_stacked_ones(dev, P, rows, dim, bs, shuffle):
    for ds in _datasets(P, rows, dim, dev):
        for drop in (False, True):
            torch.manual_seed(11)
            want = list(DataLoader(ds, batch_size=bs, shuffle=shuffle, drop_last=drop))
            after = torch.rand(1)
            torch.manual_seed(11)
            got = list(PathLoader(ds, batch_size=bs, shuffle=shuffle, drop_last=drop))
            assert torch.equal(after, torch.rand(1))
            assert len(got) == len(want)
            for (gr, gp), (wr, wp) in zip(got, want):
                assert len(gr) == len(wr)
                for g, w in zip(list(gr) + [gp], list(wr) + [wp]):
                    assert g.shape == w.shape and g.is_contiguous() and torch.equal(g, w)


@pytest.mark.gpu
def test_an_index_outside_is_refused():
    a = torch.randn(5, 3, device='cuda')
    with pytest.raises(IndexError):
        E.gather_paths([a], [0, 5])
