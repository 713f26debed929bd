"""Radial systems of the orbital correction at the sizes where the elimination can go wrong:
the smallest grids (the window of four rows is most of the matrix), counts that are no
multiple of the groups of four nodes, one column, the most columns (49), and a system whose
columns do not fit in LDS together."""
import numpy as np
import pytest

from oracle import core
from tests import systems
from tests.test_gpu_dpsi import ATOMS, _evaluate_c, _orbital_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('nrad, nang, lmax', [(5, 26, 0), (6, 26, 3), (7, 50, 1), (8, 50, 5), (9, 50, 4),
                                              (33, 110, 9), (12, 302, 24)])
def test_small_and_ragged_radial_systems(nrad, nang, lmax):
    import napmo_amd
    g, _ = systems.gpu_system(ATOMS, [[]] * 3, nrad, nang)
    o, _ = systems.oracle_system(ATOMS, [[]] * 3, nrad, nang)
    phi, ri, V = _orbital_inputs(o, 2, 11)
    doi, oi = np.array([0.03, -0.02]), np.array([-0.7, -0.4])
    d = napmo_amd.compute_dpsi(g, lmax, phi, doi, oi, ri, V, 1.0)
    for k in range(2):
        ref = core.compute_dpsi(o, lmax, phi[k], doi[k], oi[k], ri[k], V[k], 1.0, evaluate=_evaluate_c)
        scale, err = np.abs(ref).max(), np.abs(d[k] - ref).max()
        print('dpsi %d x %d lmax %d: max|d| %.3e max|err| %.3e' % (nrad, nang, lmax, scale, err))
        assert err < 1e-10 * scale


def test_columns_in_two_passes():
    # 450 radial points, lmax 8: 900 rows of 25 doubles (180 KB). Both sides solve the
    # same matrix by elimination with pivoting; its condition grows as the square of the
    # number of radial points, against 1e-10 at 300 points
    import napmo_amd
    nrad, nang, lmax = 450, 110, 8
    atoms = [('He', (0.0, 0.0, 0.0))]
    g, _ = systems.gpu_system(atoms, [[]], nrad, nang)
    o, _ = systems.oracle_system(atoms, [[]], nrad, nang)
    r = np.sqrt((o.points ** 2).sum(1))
    phi = np.exp(-1.7 * r) * (1.0 + 0.2 * o.points[:, 2])
    ri = 0.05 * phi * np.cos(o.points[:, 0]) + 0.01 * np.exp(-r ** 2)
    V = -2.0 / np.maximum(r, 1e-3) * phi
    d = napmo_amd.compute_dpsi(g, lmax, phi, 0.01, -0.9, ri, V, 1.0)
    ref = core.compute_dpsi(o, lmax, phi, 0.01, -0.9, ri, V, 1.0, evaluate=_evaluate_c)
    scale, err = np.abs(ref).max(), np.abs(d - ref).max()
    print('dpsi %d x %d lmax %d: max|d| %.3e max|err| %.3e' % (nrad, nang, lmax, scale, err))
    assert err < 1e-10 * (nrad / 300.0) ** 2 * scale
