"""The spherical projection over its row and column tiles: one density and several (16 and 32 rows
a workgroup, rows past the last), harmonics that fill no tile (lmax 0, 5, 9), angular grids below
one group of points and across the staged 128, against the sum in numpy. A density's projection
is the same in a batch as alone, to the last bit."""
import numpy as np
import pytest

from tests import systems
from tests.test_gpu_dpsi import ATOMS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('nrad, nang, lmax', [(7, 6, 0), (33, 26, 5), (18, 146, 9), (60, 302, 8)])
def test_potential_alone_and_in_a_batch(nrad, nang, lmax):
    import napmo_amd
    g, _ = systems.gpu_system(ATOMS, [[]] * 3, nrad, nang)
    o, _ = systems.oracle_system(ATOMS, [[]] * 3, nrad, nang)
    from oracle import core
    p = g.points
    # ndim functions give ndim (ndim + 1) / 2 densities: 55 x 60 shells x 3 centres take the
    # widest tiles, one density the narrowest
    ndim = 10
    psi = np.array([np.exp(-(0.3 + 0.1 * k) * ((p - np.array(ATOMS[k % 3][1])) ** 2).sum(1)) for k in range(ndim)])
    D = np.zeros((ndim, ndim))
    D[ndim - 1, 0] = 1.0  # K[0] = V[psi_0 psi_0] chi_0 with chi_0 = psi_9
    g.set_tuning(9, 17)   # the synthesis of one density at a time, as for one alone
    K = napmo_amd.compute_exchange_potential(g, psi, D, lmax)
    g.set_tuning(9, 0)
    V = napmo_amd.compute_coulomb(g, psi[0] * psi[0], lmax)
    assert np.array_equal(K[0], V * psi[ndim - 1])
    ref = core.compute_coulomb(o, psi[0] * psi[0], lmax)
    err, scale = np.abs(V - ref).max(), np.abs(ref).max()
    print('potential %d x %d lmax %d: max|err| %.3e (max|V| %.3e)' % (nrad, nang, lmax, err, scale))
    assert err < 1e-11 * scale
