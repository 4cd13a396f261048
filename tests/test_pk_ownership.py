"""Result arrays of the spectra keep no other array alive: a program that collects one small
array of many spectra holds only those."""
import numpy as np
import pytest

from pylians3_amd import _native as N

ATTRS = ('k1D', 'Nmodes1D', 'Pk1D', 'kpar', 'kper', 'Nmodes2D', 'Pk2D', 'k3D', 'Nmodes3D', 'Pk')


@pytest.mark.parametrize('dims', [2, 3, 64])
@pytest.mark.parametrize('F', [1, 2, 4])
def test_result_arrays_own_their_memory(dims, F):
    _, arrs, _ = N.alloc_pk_out(dims, F)
    for name, a in arrs.items():
        assert a.base is None and a.flags.owndata and a.flags.writeable, name


def _held(a):
    while a.base is not None:
        a = a.base
    return a.nbytes


@pytest.mark.gpu
def test_spectra_own_their_memory():
    import torch
    from pylians3_amd import Pk_library as PKL, batch
    g = torch.Generator(device='cuda').manual_seed(3)
    d = [torch.randn((2, 32, 32, 32), generator=g, device='cuda') for _ in range(2)]
    p = PKL.Pk(d[0][0], 100.0, 0, 'CIC', verbose=False)
    for k in ATTRS + ('Pkphase',):
        a = getattr(p, k)
        assert a.base is None and a.flags.owndata and a.ndim == (2 if k == 'Pk' else 1), k
    x = PKL.XPk([d[0][0], d[1][0]], 100.0, 0, ['CIC', 'CIC'])
    for k in ATTRS + ('XPk', 'PkX1D', 'PkX2D'):
        assert getattr(x, k).base is None, k
    # a batch hands out the columns of each realisation's own arrays (autos and crosses)
    for F in (1, 2):
        for r in batch.Pk_batch(d[:F], 100.0, 0, ('CIC',) * F):
            for k in ATTRS + (('Pkphase',) if F == 1 else ('XPk', 'PkX1D', 'PkX2D')):
                a = getattr(r, k)
                assert _held(a) <= (1 if F == 1 else 3) * a.nbytes, k
    assert np.array_equal(p.Pk, batch.Pk_batch(d[:1], 100.0, 0, ('CIC',))[0].Pk)
