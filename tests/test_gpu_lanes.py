"""Lane groups of the voxel-order kernels at the row lengths where they can go wrong: one, two and a
full vector of elements per lane (the narrow rows' choice where there are heavy voxels), a last
vector that overlaps its neighbour's, rows shorter than a vector, lane groups that straddle
wavefronts, two column blocks, and heavy voxels (whose atomics must count a shared element
once) at each of them.  Same bars as test_gpu_parity."""
import pytest
import torch

from tests.test_gpu_parity import run_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("C", [1, 2, 3, 4, 5, 6, 9, 11, 16, 20, 21, 24, 32, 35, 40, 41, 63, 65, 67, 85, 131, 255, 261, 341])
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


@pytest.mark.parametrize("N,C,dtype", [(270_000, 3, torch.float32), (600_000, 4, torch.float16),
                                       (1_100_000, 2, torch.float32), (1_100_000, 13, torch.bfloat16)])
def test_narrow_rows_with_heavy_voxels_in_large_tiles(N, C, dtype):
    """Tiles of 300 to 2048 positions: heavy voxels that fill many tiles, lie inside one, and end at a
    tile's edge, between ordinary ones."""
    g = torch.Generator().manual_seed(N + C)
    cnts = torch.cat([torch.randint(1, 12, (N // 12,), generator=g), torch.tensor([4096, 4095, 4097, 65, 97, 64, 30_000]),
                      torch.randint(65, 2000, (40,), generator=g)])
    cnts = cnts[torch.randperm(cnts.numel(), generator=g)]
    cnts = torch.cat([cnts, torch.ones(max(0, N - int(cnts.sum())), dtype=torch.long)])
    inv = torch.repeat_interleave(torch.arange(cnts.numel()), cnts)
    inv = inv[torch.randperm(inv.numel(), generator=g)]
    feats = torch.randn((inv.numel(), C), generator=g)
    data = run_case(f"narrow{N}", feats, inv, cnts, dtype=dtype)
    assert data.num_heavy >= 40
