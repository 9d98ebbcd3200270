"""GridHash of voxel coordinates: the occupancy-map index against the sort of the keys (both
routes, both integer types), at grids of a word's edge, dense and sparse occupancy, tables from
one slot to more tiles than one workgroup adds up, and coordinates outside the built grid."""
import numpy as np
import pytest
import torch

import torchex_amd as T

pytestmark = pytest.mark.gpu


def _check(coors, probes):
    h = T.GridHash(coors.cuda(), debug=True)
    dims = (coors.long().amax(0) + 1).tolist()
    assert list(h.dim_size) == dims
    flat = (coors[:, 0].long() * dims[1] + coors[:, 1]) * dims[2] + coors[:, 2]
    unq, inv = np.unique(flat.numpy(), return_inverse=True)
    assert np.array_equal(h.probe(coors.cuda()).cpu().numpy(), inv)
    size = 1
    while size < unq.size:
        size *= 2
    table, mask = h.table.cpu().numpy(), h.valid_mask.cpu().numpy()
    assert table.shape == (size, 2) and mask.dtype == np.bool_ and mask.sum() == unq.size
    assert h.table.dtype == torch.int32 and h.valid_table.dtype == torch.int32
    assert np.array_equal(mask, table[:, 0] != -1)
    assert np.array_equal(h.valid_table.cpu().numpy(), table[mask])
    order = np.argsort(table[mask][:, 1])
    assert np.array_equal(table[mask][order], np.stack([unq, np.arange(unq.size)], 1))
    # coordinates that were never built; a key outside the grid may meet a built one's, as in the reference
    p = (probes[:, 0] * (dims[1] * dims[2]) + probes[:, 1] * dims[2] + probes[:, 2]).int().numpy()
    at = np.searchsorted(unq, p).clip(max=unq.size - 1)
    assert np.array_equal(h.probe(probes.cuda()).cpu().numpy(), np.where(unq[at] == p, at, -1))


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("n,dims", [(1, (1, 1, 1)), (2, (1, 4, 8)), (40, (3, 11, 1)), (5000, (16, 16, 16)),
                                    (5000, (300, 300, 30)), (100, (200, 50, 40)), (9000, (1000, 1000, 60)),
                                    (3_000_000, (200, 200, 160))])
def test_index_of_coordinates(n, dims, dtype):
    g = torch.Generator().manual_seed(n)
    hi = torch.tensor(dims)
    coors = (torch.rand((n, 3), generator=g) * hi).to(dtype)
    probes = ((torch.rand((n // 2 + 3, 3), generator=g) * (hi + 2)).to(dtype) - 1)
    _check(coors, probes)
    # every second row of a wider tensor: not contiguous
    wide = torch.stack([coors, coors], 1).reshape(-1, 6).cuda()[:, :3]
    assert torch.equal(T.GridHash(wide).probe(wide), T.GridHash(coors.cuda()).probe(coors.cuda()))


def test_negative_and_oversized_coordinates_are_refused():
    with pytest.raises(RuntimeError):
        T.GridHash(torch.tensor([[3, 3, 3], [0, 0, -1]]).cuda())
    with pytest.raises(RuntimeError):
        T.GridHash(torch.tensor([[-3, -3, -3]]).int().cuda())
    with pytest.raises(AssertionError):
        T.GridHash(torch.tensor([[70_000, 70_000, 3]]).cuda())
