"""Grid hash keys that share one probe sequence: keys equal modulo the table's size start in the same slot and
step alike, so that the n-th one has to pass n - 1 taken slots.  Lengths on either side of what a lane
looks at by itself (17 slots), of the 64 more a wave looks at at once, and a table that is full."""
import numpy as np
import pytest
import torch

import torchex_amd as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shuffled", [False, True])
@pytest.mark.parametrize("n", [1, 2, 17, 18, 19, 80, 81, 82, 146, 1000, 4096])
def test_keys_of_one_sequence(n, shuffled):
    size = 1 << max(0, (n - 1).bit_length())
    rng = np.random.default_rng(n)
    keys = (5 % size + size * np.arange(2 * n)).astype(np.int32)
    if shuffled:
        rng.shuffle(keys)
    values = rng.permutation(n).astype(np.int32)
    table = T.grid_hash_build(torch.from_numpy(keys[:n]).cuda(), torch.from_numpy(values).cuda())
    assert table.shape == (size, 2)
    host = table.cpu().numpy()
    used = host[:, 0] != -1
    assert used.sum() == n and dict(host[used].tolist()) == dict(zip(keys[:n].tolist(), values.tolist()))
    # present ones, absent ones of the same sequence, and absent ones that start elsewhere, mixed
    asked = np.concatenate([keys, keys[:n] ^ 1, [-1]]).astype(np.int32)
    order = rng.permutation(asked.size)
    known = dict(zip(keys[:n].tolist(), values.tolist()))
    got = T.grid_hash_probe(torch.from_numpy(asked[order]).cuda(), table).cpu().numpy()
    assert np.array_equal(got, [known.get(int(k), -1) for k in asked[order]])


def test_a_frames_columns():
    """A grid whose strides fall badly on the table's size, built and probed through ``GridHash``."""
    g = torch.Generator().manual_seed(0)
    coors = torch.stack([torch.randint(0, 748, (90_000,), generator=g), torch.randint(0, 748, (90_000,), generator=g),
                         torch.randint(0, 30, (90_000,), generator=g)], dim=1).int()
    near = coors // torch.tensor([20, 1, 1]).int()          # whole columns side by side
    near[0] = torch.tensor([747, 747, 29])
    unq, inv = torch.unique(near, dim=0, return_inverse=True)
    table = T.GridHash(near.cuda())
    assert torch.equal(table.probe(near.cuda()).cpu().long(), inv)
    assert len(table.valid_table) == len(unq)


def test_a_grid_of_many_tiles():
    """So large a grid that its tiles of cells are scanned before they are read."""
    g = torch.Generator().manual_seed(1)
    coors = torch.randint(0, 410, (1_200_000, 3), generator=g).int()
    coors[0] = 409
    key = (coors[:, 0].long() * 410 + coors[:, 1]) * 410 + coors[:, 2]
    unq, inv = torch.unique(key, return_inverse=True)
    table = T.GridHash(coors.cuda())
    assert torch.equal(table.probe(coors.cuda()).cpu().long(), inv)
    kept = table.valid_table.cpu().long()
    assert torch.equal(torch.sort(kept[:, 0])[0], unq) and torch.equal(unq[kept[:, 1]], kept[:, 0])
