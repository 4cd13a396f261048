"""GPU tests of the column deposit (segments of tiles along z, carried planes): sparse and
clumped inputs that leave tiles of a column empty, even and uneven tile extents, one and
several tiles per segment.  An overwritten grid has the bits of an accumulated zero grid, an
accumulated one those of one float32 addition per cell, and a realisation's bits do not
depend on how its columns are cut into segments.  (Against the oracle: test_gpu_ma.py.)"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _clumps(rng, n, dims, box, cells):
    """n particles in `cells` random cells (many empty tiles), some on the box's faces."""
    c = rng.integers(0, dims, (cells, 3))
    p = (c[rng.integers(0, cells, n)] + rng.random((n, 3))) * (box / dims)
    p[: n // 20, 2] = 0.0
    p[n // 20: n // 10, 2] = np.nextafter(np.float32(box), np.float32(0))
    return np.minimum(p.astype(np.float32), np.nextafter(np.float32(box), np.float32(0)))


# (dims, particles, cells): one segment of several tiles per column needs 2048 segments and
# more (256^3: two tiles each; 400^3 uneven: four), the small grids one tile each
CASES = [(32, 300, 5), (32, 20000, 32 ** 3), (40, 500, 7), (100, 30000, 60), (256, 40000, 200),
         (256, 200000, 256 ** 3), (400, 100000, 500)]


@pytest.mark.parametrize('mas', ['CIC', 'TSC', 'PCS'])
@pytest.mark.parametrize('dims,n,cells', CASES)
def test_column_overwrite_and_accumulate(mas, dims, n, cells):
    import torch
    from pylians3_amd import MAS_library as MASL
    rng = np.random.default_rng(dims + n)
    box = 500.0
    pos = _clumps(rng, n, dims, box, cells)
    W = np.exp(rng.standard_normal(n)).astype(np.float32) if cells % 2 else None
    p = torch.from_numpy(pos).cuda()
    w = None if W is None else torch.from_numpy(W).cuda()
    g = torch.zeros((dims,) * 3, device='cuda')
    MASL.MA(p, g, box, mas, W=w)
    total = n if W is None else float(W.astype(np.float64).sum())
    assert abs(float(g.double().sum()) - total) <= 1e-5 * total
    # overwrite: the same bits, also over garbage and in cells nothing reaches
    o = torch.full((dims,) * 3, 7.0, device='cuda')
    MASL.MA_rsd(p, torch.zeros_like(p), o, box, 100.0, 0.0, 0, mas, W=w, overwrite=True)
    assert torch.equal(o, g)
    # accumulate onto a filled grid: one float32 addition per cell
    a = torch.full((dims,) * 3, 3.0, device='cuda')
    MASL.MA(p, a, box, mas, W=w)
    assert torch.equal(a, g + 3.0)


@pytest.mark.parametrize('mas', ['CIC', 'TSC', 'PCS'])
def test_column_segments_do_not_change_bits(mas):
    """A realisation alone (one tile per segment) and in a batch large enough for longer
    segments, with empty realisations and columns among them."""
    import torch
    from pylians3_amd import MAS_library as MASL, batch
    rng = np.random.default_rng(4)
    dims, box, R = 64, 100.0, 130                     # 130 * 64 tiles: segments of two
    counts = rng.integers(0, 4000, R)
    counts[3] = counts[50] = 0
    offs = np.concatenate([[0], np.cumsum(counts)]).astype(np.int64)
    pos = torch.from_numpy(np.concatenate([_clumps(rng, int(c), dims, box, 9) if c else np.zeros((0, 3), np.float32)
                                           for c in counts])).cuda()
    grids = torch.empty((R,) + (dims,) * 3, device='cuda')
    batch.MA_batch(pos, offs, grids, box, mas, accumulate=False)
    for r in (0, 3, 17, 50, 129):
        g = torch.zeros((dims,) * 3, device='cuda')
        MASL.MA(pos[int(offs[r]):int(offs[r + 1])].contiguous(), g, box, mas)
        assert torch.equal(g, grids[r])
