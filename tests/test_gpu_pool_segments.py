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
