"""Result arrays of a spectrum: one block, every array at the address its struct field holds."""
import ctypes

import numpy as np
import pytest

from pylians3_amd import _native as N


@pytest.mark.parametrize('dims', [2, 3, 65, 128])
@pytest.mark.parametrize('F', [1, 2, 4])
def test_alloc_pk_out(dims, F):
    s = N.pk_sizes(dims, F)
    S = F + F * (F - 1) // 2
    shapes = dict(k1D=(s.n1d,), Nmodes1D=(s.n1d,), Pk1D=(s.n1d, S), kpar=(s.n2d,), kper=(s.n2d,),
                  Nmodes2D=(s.n2d,), Pk2D=(s.n2d, S), k3D=(s.n3d,), Nmodes3D=(s.n3d,),
                  Pk3D=(s.n3d, 3, S), Pkphase=(s.n3d,))
    pairs = [N.alloc_pk_out(dims, F) for _ in range(2)]
    spans = []
    for out, arrs, nspec in pairs:
        assert nspec == S and list(arrs) == list(shapes)
        for name, a in arrs.items():
            assert a.shape == shapes[name] and a.dtype == np.float64 and a.flags.c_contiguous
            assert ctypes.addressof(getattr(out, name).contents) == a.ctypes.data
            spans.append((a.ctypes.data, a.ctypes.data + a.nbytes))
        assert not arrs['Pkphase'].any()
    spans.sort()                                      # no two arrays share an element
    assert all(a[1] <= b[0] for a, b in zip(spans, spans[1:]))
