"""GPU tests of segments that hold much of the particles: the column deposit cuts them into
their tiles, among segments that stay whole.  Node by node against exact sums, and a
realisation's bits alone (one tile per segment) and in a batch that cuts some of its segments."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

STENCIL = {'CIC': {0: 0.5, 1: 0.5}, 'TSC': {-1: 0.125, 0: 0.75, 1: 0.125}}


def _beam(g, n, dims, lo, hi, zlo, zhi):
    import torch
    c = torch.randint(lo, hi, (n, 3), generator=g, device='cuda')
    c[:, 2] = torch.randint(zlo, zhi, (n,), generator=g, device='cuda')
    return c


# 256^3: two tiles a segment, 400^3 (uneven): four, 512^3: sixteen; the particles of the last
# of each also take the capacity slots (256 per tile on average and more)
@pytest.mark.parametrize('dims,nbeam,nbg', [(256, 60000, 3000), (256, 700000, 500000), (400, 300000, 20000),
                                            (512, 400000, 0), (512, 3000000, 6000000)])
@pytest.mark.parametrize('mas', ['CIC', 'TSC'])
def test_beam_exact(dims, nbeam, nbg, mas):
    """Cells' corners (TSC) or middles (CIC): every contribution is a multiple of 2^-9 and
    every cell's sum below 2^15, so that float32 holds them exactly."""
    import torch
    from pylians3_amd import MAS_library as MASL
    g = torch.Generator(device='cuda').manual_seed(dims + nbeam)
    parts = [_beam(g, nbeam, dims, 30, 62, 0, dims),                          # a beam over z
             _beam(g, nbeam // 4, dims, dims - 20, dims, dims // 2, dims)]    # part of one, over the edge
    if nbg:
        parts.append(torch.randint(0, dims, (nbg, 3), generator=g, device='cuda'))
    c = torch.cat(parts)
    c = c[torch.argsort(c[:, 0] // 16)]
    pos = (c.float() + (0.5 if mas == 'CIC' else 0.0)).contiguous()
    ref = torch.bincount((c[:, 0] * dims + c[:, 1]) * dims + c[:, 2], minlength=dims ** 3).float().view((dims,) * 3)
    assert float(ref.max()) < 2 ** 15
    for ax in range(3):
        ref = sum(w * torch.roll(ref, s, ax) for s, w in STENCIL[mas].items())
    for rep in range(2):                              # the second call may take another sort
        grid = torch.zeros((dims,) * 3, device='cuda')
        MASL.MA(pos, grid, float(dims), mas)
        assert torch.equal(grid, ref)
    MASL.MA(pos, grid, float(dims), mas)              # onto a filled grid
    assert torch.equal(grid, 2 * ref)
    over = torch.full((dims,) * 3, 7.0, device='cuda')
    MASL.MA_rsd(pos, torch.zeros_like(pos), over, float(dims), 100.0, 0.0, 0, mas, overwrite=True)
    assert torch.equal(over, ref)


# segments of 2 tiles (64^3: 4 tiles a column), of 5 and 5 (160^3), of 4 and 3 uneven ones (100^3)
@pytest.mark.parametrize('dims,R', [(64, 130), (160, 17), (100, 25)])
@pytest.mark.parametrize('mas', ['CIC', 'TSC', 'PCS'])
@pytest.mark.parametrize('weighted', [False, True])
def test_cut_segments_do_not_change_bits(dims, R, mas, weighted):
    import torch
    from pylians3_amd import MAS_library as MASL, batch
    g = torch.Generator(device='cuda').manual_seed(9)
    box = 100.0
    counts = [int(x) for x in np.random.default_rng(2).integers(0, 3000, R)]
    counts[0], counts[5], counts[R // 2], counts[R - 1] = 60000, 0, 90000, 30000
    pos = []
    for r, n in enumerate(counts):
        p = torch.rand((n, 3), generator=g, device='cuda') * box
        if n >= 30000:                                # a column of tiles or two, or half of it
            p[:, :2] = p[:, :2] * 0.2 + 26.0
            if r == R - 1:
                p[:, 2] = p[:, 2] * 0.4 + 58.0
        pos.append(p)
    offs = np.concatenate([[0], np.cumsum(counts)]).astype(np.int64)
    allp = torch.cat(pos).contiguous()
    W = torch.rand(len(allp), generator=g, device='cuda') + 0.5 if weighted else None
    for accumulate in (False, True):
        grids = torch.full((R,) + (dims,) * 3, 3.0, device='cuda')
        batch.MA_batch(allp, offs, grids, box, mas, W=W, accumulate=accumulate)
        for r in (0, 1, 5, 6, R // 2, R // 2 + 1, R - 2, R - 1):
            a, b = int(offs[r]), int(offs[r + 1])
            one = torch.full((dims,) * 3, 3.0 if accumulate else 0.0, device='cuda')
            MASL.MA(allp[a:b].contiguous(), one, box, mas, W=None if W is None else W[a:b].contiguous())
            assert torch.equal(grids[r], one), (r, accumulate)


def test_cut_segments_in_a_graph():
    """Replays with other particles in the same places: units are found anew by every replay."""
    import torch
    from pylians3_amd import batch
    g = torch.Generator(device='cuda').manual_seed(4)
    dims, box, R, n = 64, 100.0, 70, 300000            # 4480 tiles: segments of two
    offs = torch.arange(R + 1, dtype=torch.int64, device='cuda') * (n // R)
    offs[1:] += n - n // R * R
    pos = torch.rand((n, 3), generator=g, device='cuda') * box
    graph = batch.BatchGraph([dict(pos=pos, offs=offs, W=None, mas='CIC')], R, dims, box)
    for rep in range(3):
        p = torch.rand((n, 3), generator=g, device='cuda') * box
        if rep:                                         # beams in all realisations, in the first ones
            m = n if rep == 1 else n // 4
            p[:m, :2] = p[:m, :2] * 0.1 + 10.0 * rep
        pos.copy_(p)
        torch.cuda.synchronize()
        graph.run()
        ref = torch.empty((R,) + (dims,) * 3, device='cuda')
        batch.MA_batch(p, offs.cpu().numpy(), ref, box, 'CIC', accumulate=False)
        assert torch.equal(graph.grids[0], ref), rep
    graph.close()
