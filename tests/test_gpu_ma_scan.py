"""GPU tests of the tile sort's offsets: the scan in one launch and in three, at the last and
first sizes of each (4096 keys a workgroup, 16 workgroups in one launch), and the small
chunks of small grids with a remainder.  NGP counts are whole numbers: exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# 32^3 grids have 8 tiles each; realisations on both sides of one scan workgroup (512 grids),
# of its last element, and of the single-launch limit (8192 grids)
@pytest.mark.parametrize('R', [1, 511, 512, 513, 8192, 8193])
def test_scan_sizes(R):
    import torch
    from pylians3_amd import batch
    rng = np.random.default_rng(R)
    dims = 32
    counts = rng.integers(0, 40, R)
    counts[-1] = 5000
    offs = np.concatenate([[0], np.cumsum(counts)]).astype(np.int64)
    n = int(offs[-1])
    cell = rng.integers(0, dims, (n, 3))
    pos = torch.from_numpy(cell.astype(np.float32)).cuda()
    grids = torch.empty((R,) + (dims,) * 3, device='cuda')
    batch.MA_batch(pos, offs, grids, float(dims), 'NGP', accumulate=False)
    real = np.repeat(np.arange(R), counts)
    flat = ((real * dims + cell[:, 0]) * dims + cell[:, 1]) * dims + cell[:, 2]
    ref = torch.bincount(torch.from_numpy(flat).cuda(), minlength=R * dims ** 3)
    assert torch.equal(grids.reshape(-1), ref.to(torch.float32))


# chunks of 1024 particles (8^3 tiles and fewer), of 8 per tile, and of 8192
@pytest.mark.parametrize('dims,axes', [(16, 3), (64, 3), (100, 3), (128, 3), (200, 3), (512, 2)])
@pytest.mark.parametrize('n', [1, 1023, 1025, 100001])
def test_small_chunks(dims, axes, n):
    import torch
    from pylians3_amd import MAS_library as MASL
    rng = np.random.default_rng(dims + n)
    cell = rng.integers(0, dims, (n, axes))
    pos = torch.from_numpy(cell.astype(np.float32)).cuda()
    g = torch.zeros((dims,) * axes, device='cuda')
    MASL.MA(pos, g, float(dims), 'NGP')
    flat = np.ravel_multi_index(tuple(cell.T), (dims,) * axes)
    ref = torch.bincount(torch.from_numpy(flat).cuda(), minlength=dims ** axes)
    assert torch.equal(g.reshape(-1), ref.to(torch.float32))
