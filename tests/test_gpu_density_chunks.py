"""The density of the resident orbitals around the number of partial sums it is
formed in (32): fewer orbitals, as many, one more, and counts that leave the last
partial short, on grids that are no multiple of a block's 256 points.

Tolerance: a sum of at most 100 positive FP64 terms in another order, 100 * 1.1e-16
relative per point; complex64 orbitals are read back as the values that are summed.
"""
import numpy as np
import pytest

from salmon_amd import gpu, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [gpu.FP64, gpu.MIXED])
@pytest.mark.parametrize("N,nk,nb", [((8, 9, 10), 1, 1), ((8, 8, 8), 2, 16), ((9, 9, 9), 1, 33), ((11, 8, 13), 5, 13),
                                     ((8, 8, 8), 4, 25)])
def test_density_matches_sum(N, nk, nb, prec):
    s = synth.make_system(N=N, L=tuple(0.64 * n for n in N), nk3=(nk, 1, 1), NB=nb, seed=8, atoms="random", natoms=1)
    s.occ = np.random.default_rng(9).uniform(0.1, 2.0, s.occ.shape)
    print(f"[gpu] density {N} {nk} x {nb}", flush=True)
    with gpu.Context(s, prec) as c:
        rho = c.psi_rho_RT()
        z = np.asarray(c.get_orbitals()).astype(np.complex128)
    ref = np.einsum("kb,kbp->p", s.occ, z.real ** 2 + z.imag ** 2)
    assert np.max(np.abs(rho - ref) / ref) < 100 * 1.1e-16
