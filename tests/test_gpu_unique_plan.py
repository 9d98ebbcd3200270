"""ScatterData straight from keys by occupancy map, whose number of voxels stays on the device until
the plan is done (up to 2^20 rows; counted first beyond), against numpy and against ScatterData of the
unique's ids: one voxel to as many as rows, ids of up to 11 bits and beyond, voxels of many slices,
crowded buckets that the bucket kernels leave to the general sequence, key bounds at a word's edge,
on either side of the map's limit, and row numbers on either side of 2^20 and of 2^22."""
import ctypes

import numpy as np
import pytest
import torch

import torchex_amd as T
from torchex_amd import _native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("n,bound,used", [
    (1, 1, 1), (5, 32, 32), (5, 33, 2), (700, 1 << 25, 700), (3000, 4096, 4096), (4000, 1 << 25, 1),
    (20_000, (1 << 25) + 1, 20_000), (60_000, 1 << 24, 1 << 24), (400_000, 1 << 20, 3), (400_000, 1 << 20, 5000),
    (4_300_000, 1 << 22, 1 << 22), (1 << 20, 1 << 24, 700), ((1 << 20) + 1, 1 << 24, 700),
    ((1 << 20) + 1, 1 << 24, 1 << 24), (1_000_000, 1 << 23, 2000), (4_300_000, 1 << 23, 90_000),
    (1 << 21, 1 << 20, 70_000), ((1 << 21) + 1, 1 << 20, 70_000), (2_098_000, 1 << 20, 1500), (2_100_000, 3, 3),
])
def test_unique_plan(n, bound, used, dtype):
    rng = np.random.default_rng(n + bound)
    keys = rng.integers(0, used, n) * (bound // used) + (bound - 1) % (bound // used)
    keys[0] = bound - 1
    if n > 1:
        keys[-1] = 0
    _check(keys, bound, dtype)


@pytest.mark.parametrize("n,voxels,rows", [(900_000, 700, 700_000), (900_000, 2048, 500_000),
                                           (900_000, 2049, 700_000), (500_000, 60_000, 300_000)])
def test_one_voxel_owns_most_rows(n, voxels, rows):
    rng = np.random.default_rng(voxels)
    keys = rng.permutation(1 << 23)[:voxels][np.concatenate([np.full(rows, voxels // 2), np.arange(voxels),
                                                             rng.integers(0, voxels, n - rows - voxels)])]
    _check(rng.permutation(keys), 1 << 23, torch.int32)


@pytest.mark.parametrize("used,dtype", [(1500, torch.int32), (2048, torch.int64), (2049, torch.int32), (70_000, torch.int64),
                                        (1 << 20, torch.int32)])
def test_more_rows_than_are_sorted_in_tiles(used, dtype):
    """Above 2^24 rows, with the number of voxels on the device only: the host provides for ids of 20 bits,
    and a bucket is a voxel (at most 2048 of them) or many."""
    n, bound = (1 << 24) + 1, 1 << 20
    rng = np.random.default_rng(used)
    keys = rng.integers(0, used, n) * (bound // used)
    keys[0] = bound - 1
    _check(keys, bound, dtype)


def _check(keys, bound, dtype):
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
    heavy = cnt > 64
    if heavy.sum() <= 64 and cnt.max() <= 96:
        heavy[:] = False
    slot_of, listed = d.slot_of.cpu().numpy(), d.heavy_ids.cpu().numpy()
    assert np.array_equal(np.sort(listed), np.flatnonzero(heavy)) and d.num_heavy == heavy.sum()
    assert np.array_equal(slot_of[listed], np.arange(listed.size)) and (slot_of[~heavy] == -1).all()


def test_keys_outside_the_bound_are_refused():
    for bad in (-1, 1000, 1 << 40):
        keys = torch.arange(1000)
        keys[500] = bad
        with pytest.raises(RuntimeError):
            T.ScatterData.from_keys(keys.cuda(), 1000)
    with pytest.raises(RuntimeError):
        T.ScatterData.from_points(torch.tensor([[0.5, 0.5, 0.5], [9.0, 0.5, 0.5]]).cuda(), [1, 1, 1], [0, 0, 0, 2, 2, 2])


@pytest.mark.parametrize("n,voxels", [(1_000_000, 2), (1_000_000, 64), (1_000_000, 2000), (1_000_000, 5000)])
def test_few_voxels_of_a_large_grid_need_no_second_plan(n, voxels):
    """The digits of the ids are split by the voxels there are, not by the most there could be: the
    bound's split would put these into one bucket and leave the plan to the general sequence."""
    lib = _native.cabi()
    vp, i64, bound = ctypes.c_void_p, ctypes.c_int64, 1 << 24
    rng = np.random.default_rng(voxels)
    keys = rng.permutation(bound)[:voxels][rng.integers(0, voxels, n)].astype(np.int32)
    unq, inv, cnt = np.unique(keys, return_inverse=True, return_counts=True)
    lib.txs_unique_bitmap_workspace_len.restype = lib.txs_plan_workspace_len.restype = i64

    def i32(m):
        return torch.empty((m,), dtype=torch.int32, device="cuda")
    k, bws, ws = torch.from_numpy(keys).cuda(), i32(lib.txs_unique_bitmap_workspace_len(i64(bound))), \
        i32(lib.txs_plan_workspace_len(i64(n), i64(n)))
    o_inv, o_unq, perm, seg, pre, slot, heavy, stats = (i32(m) for m in (n, n, n, n, n + 1, n, n, 18))
    o_cnt = torch.empty((n,), dtype=torch.int64, device="cuda")
    rc = lib.txs_unique_plan(vp(k.data_ptr()), ctypes.c_int(0), i64(n), i64(bound), vp(0), vp(bws.data_ptr()),
                             ctypes.c_int32(64), vp(ws.data_ptr()), vp(o_inv.data_ptr()), vp(o_unq.data_ptr()),
                             vp(o_cnt.data_ptr()), vp(perm.data_ptr()), vp(seg.data_ptr()), vp(pre.data_ptr()),
                             vp(slot.data_ptr()), vp(heavy.data_ptr()), vp(stats.data_ptr()),
                             vp(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    st = stats.cpu().numpy()
    assert st[16] == unq.size and st[17] == 0 and st[8] == 0      # voxels, no key outside, no general sequence
    assert st[2] == cnt.max() and st[7] == (cnt > 64).sum()
    assert np.array_equal(o_inv.cpu().numpy(), inv) and np.array_equal(o_cnt.cpu().numpy()[:unq.size], cnt)
    assert np.array_equal(perm.cpu().numpy(), np.argsort(inv, kind="stable"))


def test_what_is_kept_per_voxel_is_bounded():
    """Up to 2^20 rows the arrays with an entry per voxel may lie in one of an entry per row (20 bytes);
    beyond that they have their own length."""
    for n, most in ((1 << 20, 20 << 20), (2_000_000, 64 * 24)):
        keys = torch.randint(0, 64, (n,), generator=torch.Generator().manual_seed(n))
        d = T.ScatterData.from_keys((keys * 200_000).cuda(), 1 << 24)
        kept = {t.untyped_storage().data_ptr(): t.untyped_storage().nbytes()
                for t in (d.unq_cnts, d.preSum, d.slot_of, d.heavy_ids)}
        assert d.num_unq == 64 and sum(kept.values()) <= most + 64


@pytest.mark.parametrize("n,bound,used", [(1 << 20, 1 << 26, 1 << 20), (4_300_000, 1 << 28, 50_000)])
def test_maps_of_many_tiles(n, bound, used):
    """The most tiles of cells whose keys are added up where the cells are read, and four times as many,
    which are scanned first."""
    rng = np.random.default_rng(n)
    keys = rng.integers(0, used, n) * (bound // used)
    keys[0], keys[1] = bound - 1, 0
    _check(keys, bound, torch.int64)


@pytest.mark.parametrize("is64", [0, 1])
def test_few_keys_of_a_map_of_scanned_tiles(is64):
    lib = _native.cabi()
    vp, i64, bound, n = ctypes.c_void_p, ctypes.c_int64, (1 << 26) + 33, 5000
    rng = np.random.default_rng(is64)
    keys = rng.integers(0, bound, n)
    keys[:2] = bound - 1, 0
    keys[100:300] = keys[0]
    unq, inv, cnt = np.unique(keys, return_inverse=True, return_counts=True)
    lib.txs_unique_bitmap_workspace_len.restype = lib.txs_plan_workspace_len.restype = i64

    def i32(m):
        return torch.full((m,), -7, dtype=torch.int32, device="cuda")
    k = torch.from_numpy(keys).to(torch.int64 if is64 else torch.int32).cuda()
    bws, ws = i32(lib.txs_unique_bitmap_workspace_len(i64(bound))), i32(lib.txs_plan_workspace_len(i64(n), i64(n)))
    o_inv, o_unq, perm, seg, pre, slot, heavy, stats = (i32(m) for m in (n, n, n, n, n + 1, n, n, 18))
    o_cnt = torch.empty((n,), dtype=torch.int64, device="cuda")
    rc = lib.txs_unique_plan(vp(k.data_ptr()), ctypes.c_int(is64), i64(n), i64(bound), vp(0), vp(bws.data_ptr()),
                             ctypes.c_int32(64), vp(ws.data_ptr()), vp(o_inv.data_ptr()), vp(o_unq.data_ptr()),
                             vp(o_cnt.data_ptr()), vp(perm.data_ptr()), vp(seg.data_ptr()), vp(pre.data_ptr()),
                             vp(slot.data_ptr()), vp(heavy.data_ptr()), vp(stats.data_ptr()),
                             vp(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    st, U = stats.cpu().numpy(), unq.size
    assert st[16] == U and st[17] == 0 and st[8] == 0 and st[2] == cnt.max() and st[7] == (cnt > 64).sum()
    assert np.array_equal(o_inv.cpu().numpy(), inv) and np.array_equal(o_unq.cpu().numpy()[:U], unq)
    assert np.array_equal(o_cnt.cpu().numpy()[:U], cnt)
    assert np.array_equal(perm.cpu().numpy(), np.argsort(inv, kind="stable"))
    assert (o_unq.cpu().numpy()[U:] == -7).all()      # nothing behind the last key


def test_points_and_their_keys_make_the_same_plan():
    g = torch.Generator().manual_seed(2)
    size, rng = [0.5, 0.4, 0.3], [-10.0, -8.0, -2.0, 10.0, 8.0, 2.0]
    for n in (1, 1000, 50_001):
        pts = torch.rand((n, 4), generator=g) * torch.tensor([19.9, 15.9, 3.9, 1.0]) + torch.tensor([-9.95, -7.95, -1.95, 0.0])
        a = T.ScatterData.from_points(pts.cuda(), size, rng)
        c = T.voxelize(pts.cuda(), size, rng)
        assert torch.equal(a.coors, c) and a.spatial_size == [40, 40, 14]
        b = T.ScatterData.from_keys((c[:, 0] * 40 + c[:, 1]) * 14 + c[:, 2], 40 * 40 * 14)
        for x, y in ((a.unq_keys, b.unq_keys), (a.unq_inv, b.unq_inv), (a.unq_cnts, b.unq_cnts), (a.preSum, b.preSum),
                     (a.seg, b.seg), (a.perm, b.perm)):
            assert (x is None and y is None) or torch.equal(x, y)
        for outside in (torch.tensor([30.0, 0, 0, 0]), torch.tensor([0, 0, -2.5, 0])):
            bad = pts.clone()
            bad[n // 2] = outside
            with pytest.raises(RuntimeError):
                T.ScatterData.from_points(bad.cuda(), size, rng)
