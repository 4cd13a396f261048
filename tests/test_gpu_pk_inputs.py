"""GPU tests of how the spectra read their input fields: in place when they can be,
through a copy otherwise (unaligned views, an input that overlaps the output), and more
fields than one row-pass launch takes.  All must give the same bits."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ATTRS = ('Pk', 'Pk1D', 'Pk2D', 'Nmodes3D')


def _field(dims, seed):
    import torch
    g = torch.Generator(device='cuda').manual_seed(seed)
    return torch.randn((dims,) * 3, generator=g, device='cuda')


def _unaligned(a):
    import torch
    v = torch.empty(a.numel() + 1, device='cuda')[1:].view(a.shape)
    assert v.data_ptr() % 8 == 4
    return v.copy_(a)


@pytest.mark.parametrize('dims', [16, 64, 30])
def test_pk_and_fft_of_unaligned_views(dims):
    import torch
    from pylians3_amd import Pk_library as PKL, batch
    a = _field(dims, 3)
    u = _unaligned(a)
    keep = u.clone()
    p, q = (PKL.Pk(x, 100.0, 1, 'CIC', verbose=False) for x in (a, u))
    for k in ATTRS + ('Pkphase',):
        assert np.array_equal(getattr(p, k), getattr(q, k), equal_nan=True), k
    assert torch.equal(PKL.FFT3Dr_f(a), PKL.FFT3Dr_f(u))
    kw = dict(scales=np.float32([1.7, 0.3]), shifts=np.float32([1.0, -2.0]))
    two = torch.stack([a, 2 * a])
    r, s = (batch.Pk_batch([x], 100.0, 0, ('TSC',), **kw) for x in (two, _unaligned(two)))
    for x, y in zip(r, s):
        for k in ATTRS:
            assert np.array_equal(getattr(x, k), getattr(y, k), equal_nan=True), k
    assert torch.equal(u, keep)


def test_fft_output_over_its_input():
    import torch
    from pylians3_amd import Pk_library as PKL, _native as N
    d = 32
    a = _field(d, 5)
    ref = PKL.FFT3Dr_f(a)
    buf = torch.empty(2 * d * d * (d // 2 + 1), device='cuda')
    buf[:d ** 3] = a.reshape(-1)
    ctx = N.Context(0)
    torch.cuda.synchronize()
    N.check(N.lib().pyl_fft_r2c(ctx.handle, buf.data_ptr(), buf.data_ptr(), d, N.PTR_DEVICE))
    assert torch.equal(torch.view_as_real(ref).reshape(-1), buf)
    ctx.close()


def test_more_fields_than_one_row_launch():
    import torch
    from pylians3_amd import Pk_library as PKL, _native as N
    d, F = 16, 10
    fields = [_field(d, 20 + f) for f in range(F)]
    x = PKL.XPk(fields, 50.0, 2, ['CIC'] * F)
    for f in range(F):
        p = PKL.Pk(fields[f], 50.0, 2, 'CIC', verbose=False)
        # autos of a pair launch: the bin sums are scaled by the pair's common bound,
        # so they agree with the single field's to the fixed-point rounding
        np.testing.assert_allclose(x.Pk[:, 0, f], p.Pk[:, 0], rtol=1e-12)
