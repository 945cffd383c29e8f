"""prepare_geometry on tables that take the bucketed transposition with the most
buckets and the largest chunks: both sides of 2,048 buckets (262,144 rows, where
a chunk's LDS changes from 32,768 edges to 22,528) and the last size it takes
(2^20 rows, 8,192 buckets).  Integer work, bit-exact."""
import pytest
import torch

import pack3d_amd as p3d

pytestmark = pytest.mark.gpu


def _reverse(nb):
    """Rows that list row j, ascending, padded with -1."""
    n, width = nb.shape
    valid = nb >= 0
    source = torch.arange(n, device=nb.device)[:, None].expand(n, width)[valid]
    target, by_target = torch.sort(nb[valid].long(), stable=True)
    degree = torch.bincount(target, minlength=n)
    out = torch.full((n, max(1, int(degree.max()))), -1, dtype=torch.int32, device=nb.device)
    slot = torch.arange(target.numel(), device=nb.device) - (degree.cumsum(0) - degree)[target]
    out[target, slot] = source[by_target].int()
    return out


@pytest.mark.parametrize("n,width", [(262143, 64), (262144, 64), (262145, 64), (300000, 128), (2 ** 20, 12), (2 ** 20, 1)])
@pytest.mark.parametrize("near", [True, False])
def test_prepare_geometry_bucket_range(gpu, n, width, near):
    """near: each row's neighbours are the rows around it (a chunk reaches one or two
    buckets); else each column is a shift of its own, so that a chunk reaches all."""
    print(f"buckets n{n} width {width} near={near}", flush=True)
    gen = torch.Generator(device=gpu).manual_seed(n + width)
    shifts = torch.arange(width, device=gpu) if near else torch.randperm(n, generator=gen, device=gpu)[:width]
    rows = torch.arange(n, device=gpu)
    nb = ((rows[:, None] + shifts) % n).int()
    nb = torch.where(torch.rand(n, width, generator=gen, device=gpu) < 0.9, nb, -1)
    blocks = torch.randperm(n, generator=gen, device=gpu)[:, None]
    got = p3d.prepare_geometry(nb, blocks, 1)
    assert torch.equal(got.neighbors, nb) and torch.equal(got.blocks, blocks.int())
    assert torch.equal(got.reverse_neighbors, _reverse(nb))
