"""ScatterData straight from keys by occupancy map, whose number of voxels stays on the device until
the plan is done, against numpy and against ScatterData of the unique's ids: one voxel to as many as
rows, ids of up to 11 bits and beyond, crowded buckets that the bucket kernels leave to the general
sequence, key bounds at a word's edge, on either side of the map's limit, and above 2^22 rows."""
import numpy as np
import pytest
import torch

import torchex_amd as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("n,bound,used", [
    (1, 1, 1), (5, 32, 32), (5, 33, 2), (700, 1 << 25, 700), (3000, 4096, 4096), (4000, 1 << 25, 1),
    (20_000, (1 << 25) + 1, 20_000), (60_000, 1 << 24, 1 << 24), (400_000, 1 << 20, 3), (400_000, 1 << 20, 5000),
    (4_300_000, 1 << 22, 1 << 22),
])
def test_unique_plan(n, bound, used, dtype):
    rng = np.random.default_rng(n + bound)
    keys = rng.integers(0, used, n) * (bound // used) + (bound - 1) % (bound // used)
    keys[0] = bound - 1
    if n > 1:
        keys[-1] = 0
    unq, inv, cnt = np.unique(keys, return_inverse=True, return_counts=True)
    d = T.ScatterData.from_keys(torch.from_numpy(keys).to(dtype).cuda(), bound)
    assert d.num_unq == unq.size and d.unq_cnts.shape == (unq.size, 1) and d.unq_cnts.dtype == torch.int64
    assert np.array_equal(d.unq_keys.cpu().numpy(), unq)
    assert np.array_equal(d.unq_inv.cpu().numpy(), inv)
    assert np.array_equal(d.unq_cnts.cpu().numpy()[:, 0], cnt)
    e = T.ScatterData(torch.from_numpy(inv).cuda(), torch.from_numpy(cnt).cuda())
    assert (d.max_cnt, d.num_heavy, d.num_special, d.is_sorted) == (e.max_cnt, e.num_heavy, e.num_special, e.is_sorted)
    for a, b in ((d.preSum, e.preSum), (d.perm, e.perm), (d.seg, e.seg)):
        assert (a is None and b is None) or torch.equal(a, b)
    assert torch.equal(d.slot_of >= 0, e.slot_of >= 0)
    assert torch.equal(d.heavy_ids.sort()[0], e.heavy_ids.sort()[0])


def test_keys_outside_the_bound_are_refused():
    for bad in (-1, 1000, 1 << 40):
        keys = torch.arange(1000)
        keys[500] = bad
        with pytest.raises(RuntimeError):
            T.ScatterData.from_keys(keys.cuda(), 1000)
    with pytest.raises(RuntimeError):
        T.ScatterData.from_points(torch.tensor([[0.5, 0.5, 0.5], [9.0, 0.5, 0.5]]).cuda(), [1, 1, 1], [0, 0, 0, 2, 2, 2])
