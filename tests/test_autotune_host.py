"""The autotuner's candidates and cache keys, on the CPU: the library's own shape is among the
candidates of every FP64 plan (else tuning can only replace it), their partial sums of F stay
small, and a choice timed on replaced kernels is not taken from the cache."""
from types import SimpleNamespace

import pytest

from napmo_amd import autotune


@pytest.mark.parametrize('n', [1, 130, 300, 480, 640, 641, 1000])
def test_default_shape_is_a_candidate(n):
    cands = autotune.candidates(SimpleNamespace(precision='fp64', nbasis=n, npoint=472000))
    assert {'fock_wg': 0} in cands
    assert 'density_ks' not in autotune.DEFAULTS and 'density_pf' not in autotune.DEFAULTS


@pytest.mark.parametrize('n', [161, 300, 480, 640])
def test_candidates_partials_stay_below_a_quarter_of_phi(n):
    # a workgroup takes up to 128 of the nb (nb + 1) / 2 blocks of one chunk, a chunk's partial is
    # 2 KB a block: with W workgroups at most 128 W x 2 KB
    nb = -(-n // 16)
    blocks = nb * (nb + 1) // 2
    strips = -(-blocks // 128)
    for c in autotune.candidates(SimpleNamespace(precision='fp64', nbasis=n, npoint=472000)):
        partial = max(1, c['fock_wg'] // strips) * blocks * 256 * 8
        assert partial <= 0.25 * 8 * 472000 * n, c


def test_choices_for_replaced_kernels_are_not_read():
    f = SimpleNamespace(precision='fp64', nbasis=300, npoint=472000)
    assert autotune.shape_key(f) != 'fp64:ld320:N524288'
    assert autotune.shape_key(f).startswith('fp64:ld320:N524288:')
