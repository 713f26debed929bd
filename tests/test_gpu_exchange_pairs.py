"""The exchange potential's pair densities and accumulation over batches of pairs: one orbital,
a second batch of two pairs that starts inside a row (11 orbitals, 66 pairs in batches of 64),
and one of 14 (12 orbitals), against the sum formed on the host from single potentials."""
import numpy as np
import pytest

from tests import systems
from tests.test_gpu_dpsi import ATOMS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('ndim', [1, 2, 11, 12])
def test_pairs_over_batches(ndim):
    import napmo_amd
    g, _ = systems.gpu_system(ATOMS, [[]] * 3, 14, 26)
    rng = np.random.default_rng(ndim)
    p = g.points
    psi = np.array([np.exp(-(0.4 + 0.1 * k) * ((p - np.array(ATOMS[k % 3][1])) ** 2).sum(1)) *
                    (1.0 + 0.3 * np.sin(k + p[:, k % 3])) for k in range(ndim)])
    D = rng.normal(size=(ndim, ndim))
    g.set_tuning(9, 17)  # every potential by itself, as compute_coulomb does
    K = napmo_amd.compute_exchange_potential(g, psi, D, 3)
    g.set_tuning(9, 0)
    chi, bound_chi = D.T @ psi, np.abs(D.T) @ np.abs(psi)
    ref, bound = np.zeros_like(psi), np.zeros_like(psi)
    for s in range(ndim):
        for v in range(s + 1):
            aux = napmo_amd.compute_coulomb(g, psi[s] * psi[v], 3)
            for a, b in ((v, s),) if s == v else ((v, s), (s, v)):
                ref[a] += aux * chi[b]
                bound[a] += np.abs(aux) * bound_chi[b]
    # chi and K are sums of ndim products on each side: at most ndim + 1 roundings of 2^-53 each
    err = np.abs(K - ref)
    print('exchange of %d: max|err| %.3e (max|K| %.3e)' % (ndim, err.max(), np.abs(ref).max()))
    assert np.all(err <= 4 * (ndim + 1) * 2.0 ** -53 * bound)
