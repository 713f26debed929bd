"""FP64 contraction Phi^T diag(w bw v) Phi over upper 16 x 16 blocks against the plain product
of the oracle's basis values, at the edges of its shapes: 1 to 4 block rows (sets of waves over
different points), 5 to 10 (4 waves per workgroup), 11 to 20 and 21 to 40 (8 waves), the last
block row partly filled or full, more than 40 block rows (64 x 64 tiles), and few points."""
import numpy as np
import pytest

from oracle import cext as ocx
from tests import systems

pytestmark = pytest.mark.gpu

ATOMS = [('O', (0.0, 0.0, 0.0)), ('H', (1.1, 0.9, 0.0)), ('N', (-1.2, 0.7, 0.6))]


def _s_shells(n):
    """n s functions of distinct exponents dealt to the three atoms."""
    per = [[], [], []]
    for k in range(n):
        per[k % 3].append({'l': 0, 'prim': [0.2 * 1.015 ** k], 'cont': [1.0]})
    return per


@pytest.mark.parametrize('n,sizes', [
    (1, 'small'), (16, 'small'), (17, 'mid'), (33, 'mid'), (48, 'small'), (49, 'mid'), (64, 'tiny'),
    (65, 'mid'), (97, 'mid'), (128, 'mid'), (129, 'mid'), (160, 'tiny'), (161, 'mid'), (191, 'mid'),
    (240, 'mid'), (300, 'mid'), (320, 'tiny'), (321, 'mid'), (369, 'mid'), (480, 'mid'), (640, 'mid'),
    (641, 'small')])
def test_block_contraction_matches_plain_product(n, sizes):
    import napmo_amd
    sz = {'tiny': [(3, 6)] * 3, 'small': [(9, 26), (7, 14), (5, 38)], 'mid': [(30, 50), (22, 110), (17, 26)]}[sizes]
    g, b = systems.gpu_system(ATOMS, _s_shells(n), None, None, sizes=sz)
    ob = _oracle_basis(n)
    f = napmo_amd.GridFock(g, b, 2, 'fp64')
    v = np.random.default_rng(n).normal(size=g.size)
    F = f.contract(v)
    phi = ocx.basis_compute(ob, g.points)
    s = g.weights * g.becke_weights * v
    ref = phi.T @ (s[:, None] * phi)
    # both are FP64 sums of N products in different orders, over the same Phi up to the last
    # bits of exp: |difference| <= (N + 64) 2^-53 sum |terms|, with N < 6,000
    bound = (g.size + 64) * 2.0 ** -53 * (np.abs(phi).T @ (np.abs(s)[:, None] * np.abs(phi))) + 1e-300
    assert np.array_equal(F, F.T)
    assert np.max(np.abs(F - ref) / bound) < 1.0


def _oracle_basis(n):
    from oracle import core
    ob = core.Basis()
    for (_, o), sh in zip(ATOMS, _s_shells(n)):
        for shell in sh:
            ob.add_shell(o, shell['l'], shell['prim'], shell['cont'])
    return ob
