"""GPU tests of the staged scatter of small 3D grids (16 M particles and more): chunks in random
order, in lattice order and both in one call, weighted or not, batches with ragged and empty
realisations.  NGP of whole weights is exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _cells(g, dims, n, order):
    import torch
    k = torch.randint(0, dims ** 3, (n,), generator=g, device='cuda')
    if order == 'sorted':
        k = k.sort()[0]
    elif order == 'mixed':
        k[: n // 2] = k[: n // 2].sort()[0]
    cell = torch.stack([k // dims ** 2, k // dims % dims, k % dims], 1)
    return cell.float().contiguous(), k


def _weights(g, n):
    import torch
    return torch.randint(1, 9, (n,), generator=g, device='cuda').float()


def _ref(k, w, dims):
    import torch
    w = None if w is None else w.double()
    return torch.bincount(k, weights=w, minlength=dims ** 3).float().view((dims,) * 3)


# 512 tiles, fewer and uneven ones, a few tiles (split deposits), 729 tiles (not staged)
@pytest.mark.parametrize('dims', [128, 100, 32, 144])
@pytest.mark.parametrize('order', ['random', 'sorted', 'mixed'])
@pytest.mark.parametrize('weighted', [False, True])
def test_staged_scatter(dims, order, weighted):
    import torch
    from pylians3_amd import MAS_library as MASL
    g = torch.Generator(device='cuda').manual_seed(dims)
    n = (16 << 20) + 4097
    cell, k = _cells(g, dims, n, order)
    W = _weights(g, n) if weighted else None
    grid = torch.zeros((dims,) * 3, device='cuda')
    MASL.MA(cell, grid, float(dims), 'NGP', W=W)
    assert torch.equal(grid, _ref(k, W, dims))


@pytest.mark.parametrize('weighted', [False, True])
def test_staged_scatter_batch(weighted):
    import torch
    from pylians3_amd import batch
    g = torch.Generator(device='cuda').manual_seed(5)
    dims, counts = 64, [1 << 20, 0, 1, 70001, 8192, 0, 16 << 20, 63]
    offs = np.concatenate([[0], np.cumsum(counts)]).astype(np.int64)
    parts = [_cells(g, dims, c, 'sorted' if i == 3 else 'random') for i, c in enumerate(counts)]
    pos = torch.cat([p[0] for p in parts])
    W = _weights(g, len(pos)) if weighted else None
    grids = torch.empty((len(counts),) + (dims,) * 3, device='cuda')
    batch.MA_batch(pos, offs, grids, float(dims), 'NGP', W=W, accumulate=False)
    for r, (_, k) in enumerate(parts):
        w = None if W is None else W[int(offs[r]):int(offs[r + 1])]
        assert torch.equal(grids[r], _ref(k, w, dims)), r
