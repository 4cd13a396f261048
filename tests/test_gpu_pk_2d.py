"""GPU tests of the 2D bins, normalised in the reduction: every axis (their order differs),
one field, a pair and three fields (several launches), odd and even sides."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('axis', [0, 1, 2])
@pytest.mark.parametrize('F', [1, 2, 3])
@pytest.mark.parametrize('dims', [16, 33, 64])
def test_2d_bins_hold_the_power_of_the_3d_ones(dims, F, axis):
    import torch
    from pylians3_amd import Pk_library as PKL
    g = torch.Generator(device='cuda').manual_seed(dims + F)
    d = [torch.randn((dims,) * 3, generator=g, device='cuda') for _ in range(F)]
    d = [x + 0.5 * d[0] for x in d]                  # correlated: cross spectra of one sign
    if F == 1:
        p = PKL.Pk(d[0], 500.0, axis, 'None', verbose=False)
        two, three = p.Pk2D[:, None], p.Pk[:, 0][:, None]
    else:
        p = PKL.XPk(d, 500.0, axis, ['None'] * F)
        two = np.concatenate([p.Pk2D, p.PkX2D], 1)
        three = np.concatenate([p.Pk[:, 0], p.XPk[:, 0]], 1)
    n2 = p.Nmodes2D[:, None]
    assert np.isnan(two[p.Nmodes2D == 0]).all() and np.isfinite(two[p.Nmodes2D > 0]).all()
    # both hold every independent mode once, the 2D bins the mean's too (all sums are exact to
    # 2^-40 of the largest mode and better; float64 from there)
    fact = (500.0 / dims ** 2) ** 3
    m = [float(x.double().sum()) for x in d]
    dc = [a * a for a in m] + [m[i] * m[j] for i in range(F) for j in range(i + 1, F)]
    total = np.nansum(two * n2, 0)
    np.testing.assert_allclose(total - np.array(dc) * fact, (three * p.Nmodes3D[:, None]).sum(0),
                               rtol=0, atol=1e-6 * float(np.abs(total).max()))
