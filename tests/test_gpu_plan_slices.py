"""Index preparation of ids that fill the bucket kernels' slices in every way: one slice or
several, voxels with a short run of rows in a slice, one at the ballots' limit (24), at the heavy
threshold (64) and a long one (up to a slice that is one voxel), few and many voxels per bucket, grouped rows, empty voxels.  The plan
is whole numbers with one right answer: a stable sort by voxel."""
import ctypes

import numpy as np
import pytest
import torch

import torchex_amd as T
from torchex_amd import _native

pytestmark = pytest.mark.gpu


def _ids(kind, U, rng):
    if kind == "even":            # short runs
        c = rng.integers(0, 6, U)
    elif kind == "edges":         # 63, 64, 65 rows, and runs of a slice's length and one off it
        c = rng.choice([0, 1, 2, 63, 64, 65, 66], U, p=[.3, .3, .3, .025, .025, .025, .025])
        c[rng.choice(U, 6, replace=False)] = [2047, 2048, 2049, 4095, 4096, 4097]
    elif kind == "long":          # long runs side by side, then as many of them in a slice as fit
        c = np.zeros(U, np.int64)
        c[U // 3:U // 3 + 200] = 65
        c[U // 3 + 200:U // 3 + 600] = 25
        c[-1] = 1
    elif kind == "limit":         # runs on either side of the ballots' limit
        c = rng.choice([0, 1, 23, 24, 25, 26], U)
    else:                         # a bucket of many slices, most of it in one voxel
        c = rng.integers(0, 3, U)
        c[U // 2] = 40_000
        c[U // 2 + 1:U // 2 + 40] = 700
    return np.repeat(np.arange(U), c)


@pytest.mark.parametrize("grouped", [False, True])
@pytest.mark.parametrize("kind", ["even", "edges", "limit", "long", "crowded"])
@pytest.mark.parametrize("U", [300, 2049, 5000, 70_000, 600_000])
def test_plan_of_slices(U, kind, grouped):
    rng = np.random.default_rng(U)
    inv = _ids(kind, U, rng)
    if not grouped:
        # long stretches of one voxel in input order too, not only shuffled rows
        rng.shuffle(inv[: inv.size // 2])
        inv[inv.size // 2:] = inv[inv.size // 2:][::-1]
    cnts = np.bincount(inv, minlength=U)
    data = T.ScatterData(torch.from_numpy(inv).cuda(), torch.from_numpy(cnts).cuda())
    order = np.argsort(inv, kind="stable")
    pre = np.concatenate([[0], np.cumsum(cnts)])
    assert np.array_equal(data.preSum.cpu().numpy(), pre)
    assert (data.perm is None) == bool((np.diff(inv) >= 0).all())
    if data.perm is not None:
        assert np.array_equal(data.perm.cpu().numpy(), order)
    seg = data.seg.cpu().numpy()
    assert np.array_equal(seg & 0x7fffffff, inv[order])
    heavy = cnts > 64
    if heavy.sum() <= 64 and cnts.max() <= 96:      # a few voxels just above the threshold stay ordinary
        heavy[:] = False
    assert data.num_heavy == heavy.sum() and data.max_cnt == cnts.max()
    # every heavy voxel owns one slot, the list's place; empty ones follow, ordinary ones own none
    listed, slot_of = data.heavy_ids.cpu().numpy(), data.slot_of.cpu().numpy()
    assert np.array_equal(np.sort(listed[:data.num_heavy]), np.flatnonzero(heavy))
    assert np.array_equal(np.sort(listed[data.num_heavy:]), np.flatnonzero(cnts == 0))
    assert np.array_equal(slot_of[listed[:data.num_heavy]], np.arange(data.num_heavy))
    assert (slot_of[cnts == 0] >= data.num_heavy).all() and (slot_of[~heavy & (cnts > 0)] == -1).all()
    assert data.num_special == heavy.sum() + (cnts == 0).sum()
    assert np.array_equal(seg < 0, heavy[inv[order]] | (cnts[inv[order]] == 0))
    # int32 ids take another first kernel than the int64 ones above
    assert data.unq_inv.dtype == torch.int32 and np.array_equal(data.unq_inv.cpu().numpy(), inv)
    same = T.ScatterData(torch.from_numpy(inv).int().cuda(), torch.from_numpy(cnts).cuda())
    assert torch.equal(same.seg, data.seg) and torch.equal(same.preSum, data.preSum)
    assert (same.perm is None and data.perm is None) or torch.equal(same.perm, data.perm)
    ranks = np.empty(inv.size, np.int64)
    ranks[order] = np.arange(inv.size) - pre[inv[order]]
    assert np.array_equal(T.ingroup_inds(torch.from_numpy(inv).cuda()).cpu().numpy(), ranks)
    assert np.array_equal(T.ingroup_inds(torch.from_numpy(inv).int().cuda()).cpu().numpy(), ranks)


def test_wrong_counts_are_refused_in_one_and_in_several_slices():
    for rows in (3000, 30_000):
        inv = torch.randint(0, 2500, (rows,), generator=torch.Generator().manual_seed(rows))
        inv[: rows // 2] = 7
        cnts = torch.bincount(inv, minlength=2500)
        cnts[7] += 1
        with pytest.raises(AssertionError):
            T.ScatterData(inv.cuda(), cnts.cuda())


@pytest.mark.parametrize("N", [400_000, (1 << 24) + 1])
def test_an_overfull_bucket_leaves_the_rows_alone(N):
    """Where one bucket holds more rows than the bucket kernels take, the call only says so: no output is
    written, and above 2^24 rows, where all rows are moved to bucket order first, nor is the space for that."""
    lib = _native.cabi()
    vp, i64 = ctypes.c_void_p, ctypes.c_int64
    U = 5000
    rng = np.random.default_rng(1)
    inv = rng.integers(0, U, N).astype(np.int32)
    inv[rng.permutation(N)[:300_000]] = 7
    ids = torch.from_numpy(inv).cuda()
    lib.txs_plan_workspace_len.restype = i64
    ws = torch.full((lib.txs_plan_workspace_len(i64(N), i64(U)),), -7, dtype=torch.int32, device="cuda")
    perm, seg, pre, slot, heavy, stats = (torch.full((n,), -7, dtype=torch.int32, device="cuda")
                                          for n in (N, N, U + 1, U, U, 16))
    rc = lib.txs_plan_build(vp(ids.data_ptr()), i64(N), i64(U), ctypes.c_int32(64), vp(0), vp(ws.data_ptr()),
                            vp(perm.data_ptr()), vp(seg.data_ptr()), vp(pre.data_ptr()), vp(slot.data_ptr()),
                            vp(heavy.data_ptr()), vp(stats.data_ptr()), vp(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    assert stats[8].item() == 1 and stats[0].item() == 1      # NEED_GENERAL, UNSORTED
    for t in (perm, seg, pre, slot, heavy) + ((ws[:2 * N],) if N > 1 << 24 else ()):
        assert (t == -7).all()


@pytest.mark.parametrize("N,U", [
    (1, 1), (2, 5000), (1023, 2), (1024, 3), (1025, 1 << 20), (3000, (1 << 22) - 1),
    (1 << 17, 1500), ((1 << 17) + 1, 1500), (350_000, 1500), (1 << 18, 700), ((1 << 18) + 1, 90_000),
    (5 << 18, 2048), ((5 << 18) + 1, 2049), (1 << 21, 1 << 20), ((1 << 21) + 1, 1_000_003),
    (1 << 24, 1 << 22), (1 << 24, 1500), ((1 << 24) + 1, 1 << 21), ((1 << 24) + 1, 1500), ((1 << 24) + 4097, 70_000)])
def test_plan_at_the_edges_of_tiles(N, U):
    """Row numbers on either side of a tile's length, of every change of it and of the most rows that are
    sorted in tiles (2^24; beyond, the rows are moved to bucket order), with few and many voxels."""
    g = torch.Generator().manual_seed(N + U)
    inv = torch.randint(0, U, (N,), generator=g)
    inv[N // 2: N // 2 + N // 8] = U // 2     # a crowded bucket, and long runs
    cnts = torch.bincount(inv, minlength=U)
    order = torch.sort(inv, stable=True)[1]
    pre = torch.cat([torch.zeros(1, dtype=torch.long), torch.cumsum(cnts, 0)])
    data = T.ScatterData(inv.cuda(), cnts.cuda())
    assert torch.equal(data.preSum.cpu().long(), pre) and data.max_cnt == int(cnts.max())
    assert (data.perm is None) == bool((inv[1:] >= inv[:-1]).all())
    assert data.perm is None or torch.equal(data.perm.cpu().long(), order)
    assert torch.equal((data.seg.cpu() & 0x7fffffff).long(), inv[order])
    ranks = torch.empty_like(inv)
    ranks[order] = torch.arange(N) - pre[inv[order]]
    assert torch.equal(T.ingroup_inds(inv.cuda()).cpu(), ranks)
    if N > 1:
        wrong = inv.clone()
        wrong[N - 1] = U
        with pytest.raises(RuntimeError):
            T.ScatterData(wrong.cuda(), cnts.cuda())
