"""Points-in-boxes pooling at the edges of its tiles, box groups and segments: hits that fill
whole words of the bit matrix, segments without any, box counts on either side of a group and
above the number whose entries an emitting workgroup adds up itself, caps that end inside a
segment.  Bit-exact against the oracle."""
import numpy as np
import pytest
import torch

import torchex_amd as T
from oracle import c_oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,P,cap,max_all", [
    (1, 1, 8, 8), (1, 1023, 5000, 5000), (2, 1025, 700, 1000), (32, 16384, 512, 50_000), (33, 16385, 3000, 60_000),
    (3, 40_001, 17_000, 60_000), (3, 40_001, 17_000, 20_001), (5, 33_000, 0, 100), (5, 33_000, 100, 1),
    (2049, 2000, 3, 50_000), (2100, 1500, 10, 700),
])
def test_pool_segments(B, P, cap, max_all):
    g = torch.Generator().manual_seed(B + P)
    rois = torch.zeros((B, 7))
    rois[:, 0] = torch.arange(B) * 3.0
    rois[:, 3:6] = 2.0 + torch.rand((B, 3), generator=g)
    rois[:, 6] = torch.rand((B,), generator=g) * 6.283
    pts = torch.rand((P, 3), generator=g) * torch.tensor([3.0 * B + 2.0, 2.0, 2.0]) - 1.0
    # one long stretch of points inside the first box, and one that is in none
    pts[: P // 2] = torch.rand((P // 2, 3), generator=g) * 0.8 + torch.tensor([-0.4, -0.4, 0.2])
    pts[P // 2: P // 2 + P // 3, 1] = 50.0
    idx, roi, feats = T.dynamic_point_pool(rois.cuda(), pts.cuda(), [0.3, 0.2, 0.1], cap, max_all)
    wi, wr, wf = orc.dynamic_point_pool(rois.numpy(), pts.numpy(), [0.3, 0.2, 0.1], cap, max_all)
    if wi.shape[0] == 0:      # the placeholder entry
        assert idx.tolist() == [-1] and roi.tolist() == [-1]
        return
    assert np.array_equal(idx.cpu().numpy(), wi) and np.array_equal(roi.cpu().numpy(), wr)
    assert np.array_equal(feats.cpu().numpy().view(np.uint32), wf.view(np.uint32))


def test_boxes_of_every_reach():
    """The grid that a group of boxes is laid on: boxes of one point, one that covers the rest, boxes far out, not
    finite or larger than the grid takes, groups of nothing but those, points on the grid's outermost sides,
    far out and not finite, and both with the samples of a batch."""
    g = torch.Generator().manual_seed(3)
    B, P = 130, 30_000
    rois = torch.zeros((B, 7))
    rois[:, :3] = torch.rand((B, 3), generator=g) * torch.tensor([100.0, 100.0, 1.0]) - torch.tensor([50.0, 50.0, 1.5])
    rois[:, 3:6] = torch.rand((B, 3), generator=g) * 5.0 + 0.5
    rois[:, 6] = torch.rand((B,), generator=g) * 6.283
    rois[3, 3:6] = 0.0
    rois[5, 3:6] = 300.0
    rois[7, 0] = 3e7
    rois[9, :2] = torch.tensor([1e6, -1e6])
    for b in range(32, 64):        # a group without a single ordinary box
        rois[b, :2] = 0.0
        rois[b, 3:6] = [1e16, 3e20, float("inf"), float("nan")][b % 4]
    rois[64, 0], rois[65, 1], rois[66, 0] = float("inf"), float("-inf"), float("nan")
    rois[67, 6] = float("nan")
    rois[96:128, 0] = 12.0         # a group on one line
    rois[128:, :2] = torch.tensor([[-2e4, 7.0], [3e4, 7.0]])
    pts = torch.rand((P, 3), generator=g) * torch.tensor([110.0, 110.0, 4.0]) - torch.tensor([55.0, 55.0, 2.0])
    pts[:130] = rois[:, :3] + torch.tensor([0.0, 0.0, 0.1])
    pts[130:260] = rois[:, :3] + rois[:, 3:6] * torch.tensor([0.5, 0.5, 0.5])
    pts[260:264] = torch.tensor([[float("nan"), 0, 0], [float("inf"), 0, 0], [0, float("-inf"), 0], [3e38, -3e38, 0]])
    pts = pts[torch.randperm(P, generator=g)]
    rb, pb = torch.randint(0, 3, (B,), generator=g), torch.randint(0, 3, (P,), generator=g)
    for mixed in (False, True):
        kw = {"rois_batch": rb.cuda(), "pts_batch": pb.cuda()} if mixed else {}
        idx, roi, feats = T.dynamic_point_pool(rois.cuda(), pts.cuda(), [0.3, 0.2, 0.1], 5000, 1_000_000, **kw)
        wi, wr, wf = orc.dynamic_point_pool(rois.numpy(), pts.numpy(), [0.3, 0.2, 0.1], 5000, 1_000_000,
                                            *((rb.numpy(), pb.numpy()) if mixed else ()))
        assert wi.shape[0] > 10_000
        assert np.array_equal(idx.cpu().numpy(), wi) and np.array_equal(roi.cpu().numpy(), wr)
        got = feats.cpu().numpy()
        assert np.array_equal(np.isnan(got), np.isnan(wf))
        assert np.array_equal(np.nan_to_num(got).view(np.uint32), np.nan_to_num(wf).view(np.uint32))


@pytest.mark.parametrize("axis", [0, 1])
@pytest.mark.parametrize("out", [-1e14, -1e10, -3e9, -5e8, -2e8, -1e6, -1e4, 1e4, 5e8, 1e14])
def test_one_box_far_out_keeps_the_others(out, axis):
    """One box of every group far out on either side, where the grid's cells are so wide that the sides of
    all other boxes fall on its end."""
    g = torch.Generator().manual_seed(5)
    B, P = 70, 8000
    rois = torch.zeros((B, 7))
    rois[:, :2] = torch.rand((B, 2), generator=g) * 100.0 - 50.0
    rois[:, 3:6] = torch.rand((B, 3), generator=g) * 5.0 + 0.5
    rois[:, 6] = torch.rand((B,), generator=g) * 6.283
    rois[[4, 40, 69], axis] = out
    pts = torch.rand((P, 3), generator=g) * torch.tensor([110.0, 110.0, 4.0]) - torch.tensor([55.0, 55.0, 2.0])
    pts[:B] = rois[:, :3] + torch.tensor([0.0, 0.0, 0.1])
    idx, roi, feats = T.dynamic_point_pool(rois.cuda(), pts.cuda(), [0.3, 0.2, 0.1], 5000, 100_000)
    wi, wr, wf = orc.dynamic_point_pool(rois.numpy(), pts.numpy(), [0.3, 0.2, 0.1], 5000, 100_000)
    assert set(wr.tolist()) == set(range(B))
    assert np.array_equal(idx.cpu().numpy(), wi) and np.array_equal(roi.cpu().numpy(), wr)
    assert np.array_equal(feats.cpu().numpy().view(np.uint32), wf.view(np.uint32))


def test_sides_at_the_ends_of_the_float_range():
    """Half a side where a float cannot hold it, sides of no extent, negative ones and the largest, with points as
    close to the box's centre and as far from it as floats go."""
    tiny, big = float(np.float32(1e-45)), float(np.finfo(np.float32).max)
    sides = [0.0, tiny, 2 * tiny, 3 * tiny, 5 * tiny, 1.0, big / 2, big, float("inf"), -1.0, -3 * tiny]
    rois = torch.zeros((3 * len(sides), 7))
    for k, s in enumerate(sides):
        for axis in range(3):
            rois[3 * k + axis, 3:6] = 2.0
            rois[3 * k + axis, 3 + axis] = s
    rois[:, 6] = -np.pi / 2       # no turn
    near = [0.0, tiny, -tiny, 2 * tiny, -2 * tiny, 3 * tiny, 0.4, -0.4, 1.1, big / 2, -big / 2, big, -big]
    pts = torch.tensor([[x, y, z] for x in near for y in near for z in near])
    for extra in ([0.0, 0.0, 0.0], [tiny, 3 * tiny, tiny], [0.5, 0.5, 0.5]):
        idx, roi, feats = T.dynamic_point_pool(rois.cuda(), pts.cuda(), extra, 3000, 200_000)
        wi, wr, wf = orc.dynamic_point_pool(rois.numpy(), pts.numpy(), extra, 3000, 200_000)
        assert wi.shape[0] > 1000
        assert np.array_equal(idx.cpu().numpy(), wi) and np.array_equal(roi.cpu().numpy(), wr)
        got = feats.cpu().numpy()
        assert np.array_equal(np.isnan(got), np.isnan(wf))
        assert np.array_equal(np.nan_to_num(got).view(np.uint32), np.nan_to_num(wf).view(np.uint32))
