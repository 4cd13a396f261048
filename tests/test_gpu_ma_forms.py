"""GPU test of the two deposit forms (a workgroup per tile, and columns of tiles): a dense PCS
realisation takes the tile form alone and the column form in a batch whose other realisations
are sparse, TSC the tile form on a small grid and the column form in a batch.  Same bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# PCS: tiles of 2048 records on average and more (64 tiles: from 131072 particles on) against
# 800; TSC: segments of four tiles and more (256 grids of 64^3)
@pytest.mark.parametrize('mas,R,n', [('PCS', 4, 131072), ('PCS', 4, 200000), ('TSC', 256, 40000)])
@pytest.mark.parametrize('weighted', [False, True])
@pytest.mark.parametrize('accumulate', [False, True])
def test_forms_give_the_same_bits(mas, R, n, weighted, accumulate):
    import torch
    from pylians3_amd import MAS_library as MASL, batch
    g = torch.Generator(device='cuda').manual_seed(R + n)
    dims, box = 64, 250.0
    counts = [n] + [1000 + r for r in range(R - 1)]
    offs = np.concatenate([[0], np.cumsum(counts)]).astype(np.int64)
    pos = torch.rand((int(offs[-1]), 3), generator=g, device='cuda') * box
    pos[: n // 3] = pos[: n // 3] * 0.3 + 100.0       # uneven tiles
    W = torch.rand(len(pos), generator=g, device='cuda') * 5 + 0.1 if weighted else None
    init = torch.rand((R,) + (dims,) * 3, generator=g, device='cuda')
    grids = init.clone()
    batch.MA_batch(pos, offs, grids, box, mas, W=W, accumulate=accumulate)
    one = init[0].clone() if accumulate else torch.zeros((dims,) * 3, device='cuda')
    MASL.MA(pos[:n].contiguous(), one, box, mas, W=None if W is None else W[:n].contiguous())
    assert torch.equal(grids[0], one)
