"""GPU tests of modes that are not counted: in the planes kz = 0 and (even sides) kz = N/2
only one mode of each conjugate pair enters the bins (Pk_library.pyx:324-327), and a caller's
half-complex field may hold anything in the other one, NaN and infinities among it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BOX = 300.0


def _field(dims, seed):
    """Whole numbers (their squares add up exactly), the largest in a counted mode."""
    rng = np.random.default_rng(seed)
    shape = (dims, dims, dims // 2 + 1)
    dk = (rng.integers(-99, 100, shape) + 1j * rng.integers(-99, 100, shape)).astype(np.complex64)
    dk[1, 1, 1] = 100 + 100j
    return dk


def _dependent(dims):
    m = dims // 2
    k = np.arange(dims)
    k = np.where(k > m, k - dims, k)
    edge = (k == 0) | ((dims % 2 == 0) & (k == m))
    skip = (k[:, None] < 0) | (edge[:, None] & (k[None, :] < 0))
    out = np.zeros((dims, dims, m + 1), bool)
    out[:, :, 0] = skip
    if dims % 2 == 0:
        out[:, :, m] = skip
    return out


@pytest.mark.parametrize('dims', [16, 17, 30, 33, 64])
@pytest.mark.parametrize('axis', [0, 1, 2])
@pytest.mark.parametrize('F', [1, 2])
def test_dependent_modes_do_not_count(dims, axis, F):
    from pylians3_amd import Pk_library as PKL
    clean = [_field(dims, 7 + f) for f in range(F)]
    dep = _dependent(dims)
    nan = [d.copy() for d in clean]
    inf = [d.copy() for d in clean]
    for a, b in zip(nan, inf):
        a[dep] = complex(np.nan, np.nan)
        b[dep] = complex(np.inf, -np.inf)
    ref, got_nan, got_inf = (PKL.Pk_from_fourier(x, BOX, dims, axis) for x in (clean, nan, inf))
    for k, v in ref.items():
        assert np.array_equal(got_nan[k], v, equal_nan=True), k
        if k != 'Pk3D':
            assert np.array_equal(got_inf[k], v, equal_nan=True), k
    # an infinite largest mode leaves the bin sums in units of 1: exact for l = 0, and each of
    # the at most Nmodes additions to a multipole's bin within 1/2
    assert np.array_equal(got_inf['Pk3D'][:, 0], ref['Pk3D'][:, 0])
    tol = 0.5 * np.array([5.0, 9.0]) * (BOX / dims ** 2) ** 3 * (1 + 1e-6)
    assert np.all(np.abs(got_inf['Pk3D'][:, 1:] - ref['Pk3D'][:, 1:]) <= tol[None, :, None])
