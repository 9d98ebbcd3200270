"""Grid hash keys that share one probe sequence: keys equal modulo the table's size start in the same slot and
step alike, so that the n-th one has to pass n - 1 taken slots.  Lengths on either side of what a lane looks at by
itself and of what a wave's lanes look at for a few keys or one, nearly full tables, and a table that is full."""
import numpy as np
import pytest
import torch

import torchex_amd as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shuffled", [False, True])
@pytest.mark.parametrize("n", [1, 2, 9, 16, 17, 18, 19, 33, 34, 63, 64, 65, 80, 81, 82, 146, 288, 1000, 4096])
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


@pytest.mark.parametrize("n,probes", [(1000, 5000), (30_000, 70_001), (65_536, 100_000), (3 << 17, 1 << 20),
                                      ((3 << 17) + 1, (1 << 20) + 1), ((1 << 20) + 1, (1 << 20) + 1)])
def test_one_long_sequence_among_many_short_ones(n, probes):
    """Numbers of keys on either side of where fewer of them get the lanes of others; 300 keys of one sequence, next to
    each other and then anywhere, among keys that find a slot soon (or, in a table that is nearly full, do not)."""
    size = 1 << (n - 1).bit_length()
    rng = np.random.default_rng(n)
    others = np.setdiff1d(rng.integers(0, 2**31 - 1, 2 * n), 5 + size * np.arange(600))
    keys = np.concatenate([5 + size * np.arange(300), rng.permutation(others)[: n - 300]]).astype(np.int32)
    for order in (np.arange(n), rng.permutation(n)):
        placed, values = keys[order], rng.permutation(n).astype(np.int32)
        table = T.grid_hash_build(torch.from_numpy(placed).cuda(), torch.from_numpy(values).cuda())
        asked = np.concatenate([placed[:probes // 2], 5 + size * np.arange(600),
                                rng.integers(0, 2**31 - 1, probes)])[:probes].astype(np.int32)
        asked = rng.permutation(asked)
        by_key = np.argsort(placed, kind="stable")
        at = np.minimum(np.searchsorted(placed[by_key], asked), n - 1)
        want = np.where(placed[by_key][at] == asked, values[by_key][at], -1)
        if n == size:     # (an absent key is looked for in every slot of a full table)
            asked, want = asked[want >= 0], want[want >= 0]
        assert np.array_equal(T.grid_hash_probe(torch.from_numpy(asked).cuda(), table).cpu().numpy(), want)
        host = table.cpu().numpy()
        assert np.array_equal(np.sort(host[host[:, 0] != -1, 0]), np.sort(placed))


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
