"""The overlap matrix keeps the order of summation of the legacy contraction (64 x 64 tiles over
the same chunks of points), to the last bit: a program orthonormalises its orbitals with it, and
orbitals that nearly span the basis magnify a change of rounding in S by many orders."""
import numpy as np
import pytest

from tests import systems
from tests.test_gpu_fock_blocks import ATOMS, _s_shells

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('n', [1, 20, 50, 65, 130, 300])
@pytest.mark.parametrize('precision', ['fp64', 'int8', 'bf16x3'])
def test_overlap_sums_as_the_legacy_contraction(n, precision):
    import napmo_amd
    from napmo_amd.wavefunction import grid_ops
    g, b = systems.gpu_system(ATOMS, _s_shells(n), None, None, sizes=[(30, 50), (22, 110), (17, 26)])
    S = napmo_amd.GridFock(g, b, 2, precision).overlap()
    phi = b.compute(g.points)
    legacy = grid_ops.compute_coupling(napmo_amd.PSIB(n), g, np.ascontiguousarray(phi.T), np.ones(g.size))
    assert np.array_equal(S, S.T)
    # the legacy contraction mirrors nothing for one operand: its upper triangle is S's
    i, j = np.triu_indices(n)
    assert np.array_equal(S[i, j], legacy[i, j])
