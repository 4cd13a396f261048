"""GPU tests of the plane pass of the FFT (sides of 64 and 128: rows and columns of a plane in
one workgroup) beside the separate passes (32, 256), and of the columns that are alone in
their group (kz = N/2)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dims', [32, 64, 128, 256])
def test_fft_against_float64(dims):
    import torch
    from pylians3_amd import Pk_library as PKL
    g = torch.Generator(device='cuda').manual_seed(dims)
    a = torch.randn((dims,) * 3, generator=g, device='cuda')
    ref = torch.fft.rfftn(a.double())
    err = PKL.FFT3Dr_f(a).to(torch.complex128) - ref
    # a radix-2^k FFT's error in the 2-norm: at most log2(n) (u + 4u (sqrt(2) + u)) of the
    # result's, u = 2^-24, here with twiddles rounded once: under 8 u log2(n)
    bound = 8 * 2.0 ** -24 * 3 * np.log2(dims) * float(ref.abs().square().sum()) ** 0.5
    assert float(err.abs().square().sum()) ** 0.5 <= bound
    # (the error of one kz column is part of it; columns of white noise share the norm)
    for kz in (0, 1, dims // 2 - 1, dims // 2):
        assert float(err[:, :, kz].abs().square().sum()) ** 0.5 <= bound / (dims // 2 + 1) ** 0.5 * 3


@pytest.mark.parametrize('dims', [64, 128])
@pytest.mark.parametrize('F', [1, 2])
def test_batch_of_planes_equals_single_cubes(dims, F):
    import torch
    from pylians3_amd import Pk_library as PKL, batch
    g = torch.Generator(device='cuda').manual_seed(F)
    R = 3
    x = [torch.randn((R,) + (dims,) * 3, generator=g, device='cuda') + f for f in range(F)]
    sc = np.exp(np.random.default_rng(1).standard_normal((R, F))).astype(np.float32)
    sh = np.arange(R * F, dtype=np.float32).reshape(R, F) / 3
    res = batch.Pk_batch(x, 100.0, 1, ('CIC', 'TSC')[:F], scales=sc, shifts=sh)
    for r in range(R):
        # (on the host: torch multiplies by a scalar's reciprocal)
        d = [torch.from_numpy(x[f][r].cpu().numpy() / sc[r, f] - sh[r, f]).cuda() for f in range(F)]
        one = (PKL.Pk(d[0], 100.0, 1, 'CIC', verbose=False) if F == 1
               else PKL.XPk(d, 100.0, 1, ['CIC', 'TSC']))
        for k in ('Pk', 'Pk1D', 'Pk2D') + (('XPk',) if F == 2 else ()):
            assert np.array_equal(getattr(res[r], k), getattr(one, k), equal_nan=True), k
