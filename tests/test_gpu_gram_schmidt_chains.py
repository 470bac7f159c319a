"""Gram-Schmidt of bands that each keep a part of their norm but depend on each
other in turn, b_j = e_{j-1} + s e_j: no single overlap or pivot is extreme, and
the whole panel is dependent to rounding (csrc/gsblock.hpp leaves such panels to
the band-by-band form).  Chains within the first panel, from its last band on in
the second, and mixed over the whole grid by a unitary; and mild chains, which
stay in panels.

Tolerances: orthonormality 1e-13 as for nearly dependent pairs.  On grid points as
the e_j the overlaps are sums of one term each, so two passes of the sequential
loop leave rounding: 1e-12.  Mild chains: eps times the condition of the panel,
below 1e4 (s = 0.1, four bands) and 1e3 (s = 0.5, six bands): 1e-11.
"""
import numpy as np
import pytest

from helpers import rel
from salmon_amd import gpu, synth

pytestmark = pytest.mark.gpu
N, NK = (9, 10, 11), 2


def system(nb, seed=3):
    s = synth.make_system(N=N, L=tuple(0.64 * n for n in N), nk3=(NK, 1, 1), NB=nb, seed=seed, atoms="random", natoms=1,
                          orbitals=False)
    rng = np.random.default_rng(seed)
    s.zu = rng.standard_normal((NK, nb, s.NL)) + 1j * rng.standard_normal((NK, nb, s.NL))
    return s


def chain(e, s):
    return np.array([e[0]] + [e[j - 1] + s * e[j] for j in range(1, len(e))])


def run(s):
    with gpu.Context(s, gpu.FP64) as c:
        c.gram_schmidt()
        return c.get_orbitals()


def overlap_error(s, z):
    o = np.einsum("kbn,kcn->kbc", z.conj(), z) * s.Hxyz
    return np.abs(o - np.eye(z.shape[1])).max()


@pytest.mark.parametrize("first", [0, 15])
@pytest.mark.parametrize("step,n", [(0.03, 12), (0.03, 8), (1e-3, 6), (1e-3, 8), (3e-4, 6)])
def test_chains_of_grid_points(step, n, first):
    """Bands first .. first + n - 1 of k point 1 are a chain of grid points; the bands below it are grid points too."""
    s = system(first + n)
    e = np.zeros((first + n, s.NL), complex)
    e[np.arange(first + n), 7 + 13 * np.arange(first + n)] = 2.5
    s.zu[1] = np.concatenate([e[:first], chain(e[first:], step)])
    z = run(s)
    print(f"[gpu] chain s={step} n={n} from band {first}: overlap error {overlap_error(s, z):.1e}", flush=True)
    assert overlap_error(s, z) < 1e-13
    assert rel(z[1], e / (2.5 * np.sqrt(s.Hxyz))) < 1e-12
    assert rel(z[0], synth.gram_schmidt(s.zu[:1], s.Hxyz)[0]) < 1e-12


@pytest.mark.parametrize("first", [0, 10, 16])
@pytest.mark.parametrize("step,n", [(0.1, 10), (0.03, 7), (0.03, 12), (1e-3, 5), (1e-3, 8), (3e-4, 6)])
@pytest.mark.parametrize("seed", range(6))
def test_chains_over_the_whole_grid(step, n, first, seed):
    s = system(first + n, seed=5)
    rng = np.random.default_rng(seed)
    e = np.linalg.qr(rng.standard_normal((s.NL, first + n)) + 1j * rng.standard_normal((s.NL, first + n)))[0].T
    s.zu[0] = np.concatenate([e[:first], chain(e[first:], step)])
    z = run(s)
    print(f"[gpu] dense chain s={step} n={n} from band {first}: overlap error {overlap_error(s, z):.1e}", flush=True)
    assert overlap_error(s, z) < 1e-13


@pytest.mark.parametrize("step,n", [(0.1, 4), (0.5, 6)])
def test_mild_chains(step, n):
    s = system(n, seed=7)
    rng = np.random.default_rng(8)
    e = np.linalg.qr(rng.standard_normal((s.NL, n)) + 1j * rng.standard_normal((s.NL, n)))[0].T
    s.zu[1] = chain(e, step)
    z = run(s)
    assert overlap_error(s, z) < 1e-13
    assert rel(z, synth.gram_schmidt(s.zu, s.Hxyz)) < 1e-11


def test_other_k_points_are_left_alone():
    """A k point left to the band-by-band form changes nothing of the others: eager, captured and replayed calls."""
    s = system(9, seed=9)
    good = run(s)
    s.zu[1, 6] = s.zu[1, 2] * (0.3 + 0.9j) + 1e-6 * s.zu[1, 6]
    with gpu.Context(s, gpu.FP64) as c:
        for call in range(3):
            c.put_orbitals(s.zu)
            c.gram_schmidt()
            z = c.get_orbitals()
            assert np.array_equal(z[0], good[0]), call
            assert overlap_error(s, z) < 1e-13
        s.zu[0], s.zu[1] = s.zu[1].copy(), s.zu[0].copy()  # the replayed launches follow the flags
        c.put_orbitals(s.zu)
        c.gram_schmidt()
        z1 = c.get_orbitals()
        assert np.array_equal(z1[1], good[0]) and np.array_equal(z1[0], z[1])
