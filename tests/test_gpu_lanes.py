"""Lane groups of the voxel-order kernels at the row lengths where they can go wrong: a last
vector that overlaps its neighbour's, rows shorter than a vector, lane groups that straddle
wavefronts, two column blocks, and heavy voxels (whose atomics must count a shared element
once) at each of them.  Same bars as test_gpu_parity."""
import pytest
import torch

from tests.test_gpu_parity import run_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("C", [2, 3, 5, 6, 9, 11, 21, 63, 65, 67, 85, 131, 255, 261, 341])
def test_rows_that_fill_no_whole_vectors(C, dtype):
    g = torch.Generator().manual_seed(1000 + C)
    cnts = torch.cat([torch.randint(1, 12, (400,), generator=g), torch.randint(65, 400, (9,), generator=g),
                      torch.tensor([0, 0, 64, 97])])
    inv = torch.repeat_interleave(torch.arange(cnts.numel()), cnts)
    inv = inv[torch.randperm(inv.numel(), generator=g)]
    feats = torch.randn((inv.numel(), C), generator=g)
    feats[torch.rand(feats.shape, generator=g) < 0.05] = 1.25    # ties
    data = run_case(f"vectors{C}", feats, inv, cnts, dtype=dtype)
    assert data.num_heavy == 10
