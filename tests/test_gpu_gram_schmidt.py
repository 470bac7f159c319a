"""Gram-Schmidt of the resident orbitals (panels of 16 bands, csrc/gsblock.hpp)
against the sequential loop in NumPy: band counts around the panel, grids that
are no multiple of a block's points, several k points, bands that nearly depend
on each other (which the panels leave to the band-by-band form) and a band that
is not finite.

Tolerances: a band's component along the others is known to the rounding eps of
the overlaps over the sine of the angle it keeps to them.  Random bands keep
angles near one: 1e-12.  Sines of 1e-3 and 1e-5 leave 1e-13 and 1e-11 times the
growth of a few bands' sums: 1e-10 and 1e-8.  Complex64 contexts round the
result to single: 1e-6.
"""
import numpy as np
import pytest

from helpers import rel
from salmon_amd import gpu, synth

pytestmark = pytest.mark.gpu


def system(N, nk, nb, seed=3):
    s = synth.make_system(N=N, L=tuple(0.64 * n for n in N), nk3=(nk, 1, 1), NB=nb, seed=seed, atoms="random", natoms=1,
                          orbitals=False)
    rng = np.random.default_rng(seed)
    s.zu = rng.standard_normal((nk, nb, s.NL)) + 1j * rng.standard_normal((nk, nb, s.NL))
    return s


def orthonormal(s, prec=gpu.FP64):
    with gpu.Context(s, prec) as c:
        c.gram_schmidt()
        return c.get_orbitals()


@pytest.mark.parametrize("nb", [1, 2, 15, 16, 17, 32, 41])
@pytest.mark.parametrize("N,nk", [((8, 8, 8), 3), ((9, 9, 9), 1), ((9, 10, 11), 2), ((13, 8, 21), 1)])
def test_panels_match_the_sequential_loop(N, nk, nb):
    s = system(N, nk, nb)
    z = orthonormal(s)
    assert rel(z, synth.gram_schmidt(s.zu, s.Hxyz)) < 1e-12
    o = np.einsum("kbn,kcn->kbc", z.conj(), z) * s.Hxyz
    assert np.abs(o - np.eye(nb)).max() < 1e-14 * 16


@pytest.mark.parametrize("sine,tol", [(1e-3, 1e-10), (1e-5, 1e-8)])
@pytest.mark.parametrize("i,j", [(3, 9), (2, 20), (17, 18)])
def test_nearly_dependent_bands(sine, tol, i, j):
    """Band j close to band i: within one panel, across panels, and in the second panel."""
    s = system((9, 10, 11), 2, 21)
    s.zu[1, j] = s.zu[1, i] * (0.7 - 0.4j) + sine * s.zu[1, j]
    z = orthonormal(s)
    assert rel(z, synth.gram_schmidt(s.zu, s.Hxyz)) < tol
    o = np.einsum("kbn,kcn->kbc", z.conj(), z) * s.Hxyz
    assert np.abs(o - np.eye(21)).max() < 1e-13


def test_bands_that_are_not_finite():
    s = system((8, 8, 8), 2, 18)
    good = orthonormal(s)
    s.zu[1, 5, 7] = np.nan
    z = orthonormal(s)
    assert rel(z[0], good[0]) < 1e-12 and rel(z[1, :5], good[1, :5]) < 1e-12
    assert np.isnan(z[1, 5:]).all()


def test_complex64_orbitals():
    s = system((9, 10, 11), 2, 19)
    assert rel(orthonormal(s, gpu.MIXED), synth.gram_schmidt(s.zu, s.Hxyz)) < 1e-6
