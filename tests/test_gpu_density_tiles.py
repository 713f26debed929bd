"""Density over column tiles against the plain product: P not symmetric (the fold onto the lower
block triangle takes its symmetric part), 1 to 41 blocks of 16 functions (partly filled last
blocks, odd and even numbers of 16-function groups, one to eleven 64-column tiles), and the
orbital form past 64 orbitals with 1 to 4 blocks in the last tile."""
import numpy as np
import pytest

from oracle import cext as ocx
from tests import systems
from tests.test_gpu_fock_blocks import ATOMS, _oracle_basis, _s_shells

pytestmark = pytest.mark.gpu

# Both sides form exp(-zeta r^2) from their own rounding of zeta r^2 (two units in its last place
# apart at most), and |zeta r^2| < 746 wherever the value is not zero: each of the two factors Phi
# of a term moves by up to 2 * 746 units of 2^-53.
EXP = 2 * 2 * 746


def _plan(n):
    import napmo_amd
    g, b = systems.gpu_system(ATOMS, _s_shells(n), None, None, sizes=[(30, 50), (22, 110), (17, 26)])
    return g, napmo_amd.GridFock(g, b, 2, 'fp64'), ocx.basis_compute(_oracle_basis(n), g.points)


@pytest.mark.parametrize('n', [1, 16, 17, 40, 63, 64, 65, 80, 97, 128, 130, 193, 300, 657])
def test_p_form_takes_the_symmetric_part(n):
    g, f, phi = _plan(n)
    P = np.random.default_rng(n).normal(size=(n, n))
    _, _, _, rho, _ = f.build(P, want_grid=True)
    ref = ((phi @ P) * phi).sum(1)
    # FP64 sums of n^2 products in another order; EXP: Phi itself
    bound = (2 * n + 64 + EXP) * 2.0 ** -53 * ((np.abs(phi) @ np.abs(P)) * np.abs(phi)).sum(1) + 1e-300
    assert np.max(np.abs(rho - ref) / bound) < 1.0


@pytest.mark.parametrize('n,nocc', [(70, 65), (97, 80), (128, 97), (130, 113), (193, 128), (300, 130)])
def test_orbital_form_past_one_tile(n, nocc):
    g, f, phi = _plan(n)
    C = np.random.default_rng(n).normal(size=(n, nocc))
    _, _, _, rho, _ = f.build_orbitals(C, 2.0, want_grid=True)
    ref = 2.0 * ((phi @ C) ** 2).sum(1)
    bound = (2 * n + nocc + 64 + EXP) * 2.0 ** -52 * ((np.abs(phi) @ np.abs(C)) ** 2).sum(1) + 1e-300
    assert np.max(np.abs(rho - ref) / bound) < 1.0


# From 1,024 workgroups of 256 points on, a wave takes 64 rows instead of 32: three atoms of
# 50 x 590 points (346 point tiles, 4 column tiles from 193 functions on) and of 75 x 590 (519
# point tiles, two column tiles from 65 orbitals on). The reference on every 31st point and on the
# first and last 300.
def _wide_plan(n, nrad):
    import napmo_amd
    g, b = systems.gpu_system(ATOMS, _s_shells(n), None, None, sizes=[(nrad, 590)] * 3)
    at = np.unique(np.concatenate([np.arange(300), np.arange(0, g.size, 31), np.arange(g.size - 300, g.size)]))
    return napmo_amd.GridFock(g, b, 2, 'fp64'), at, ocx.basis_compute(_oracle_basis(n), g.points[at])


@pytest.mark.parametrize('n', [193, 224, 300, 337, 657])
def test_p_form_64_rows_a_wave(n):
    f, at, phi = _wide_plan(n, 50)
    P = np.random.default_rng(n).normal(size=(n, n))
    _, _, _, rho, _ = f.build(P, want_grid=True)
    ref = ((phi @ P) * phi).sum(1)
    bound = (2 * n + 64 + EXP) * 2.0 ** -53 * ((np.abs(phi) @ np.abs(P)) * np.abs(phi)).sum(1) + 1e-300
    assert np.max(np.abs(rho[at] - ref) / bound) < 1.0


@pytest.mark.parametrize('n,nocc', [(66, 65), (97, 90), (130, 113), (193, 128), (300, 130), (300, 161)])
def test_orbital_form_64_rows_a_wave(n, nocc):
    f, at, phi = _wide_plan(n, 75)
    C = np.random.default_rng(n).normal(size=(n, nocc))
    _, _, _, rho, _ = f.build_orbitals(C, 2.0, want_grid=True)
    ref = 2.0 * ((phi @ C) ** 2).sum(1)
    bound = (2 * n + nocc + 64 + EXP) * 2.0 ** -52 * ((np.abs(phi) @ np.abs(C)) ** 2).sum(1) + 1e-300
    assert np.max(np.abs(rho[at] - ref) / bound) < 1.0
