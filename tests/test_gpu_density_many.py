"""The density of more orbitals than 32 partial sums take 256 each of, on grids of a
few blocks of points, where it is formed in more of them (in two stages), and beside
the line between the two, which lies at half as many blocks in FP64.

Tolerance: a sum of n positive FP64 terms in another order, n * 1.1e-16 relative.
"""
import numpy as np
import pytest

from salmon_amd import gpu, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [gpu.FP64, gpu.MIXED])
@pytest.mark.parametrize("N,nk,nb", [((8, 8, 8), 128, 64), ((8, 8, 8), 129, 66), ((8, 9, 10), 400, 43), ((10, 11, 12), 129, 66),
                                     ((12, 12, 12), 129, 66),
                                     ((13, 14, 17), 129, 66)])
def test_density_of_many_orbitals(N, nk, nb, prec):
    s = synth.make_system(N=N, L=tuple(0.64 * n for n in N), nk3=(1, 1, 1), NB=1, seed=8, atoms="random", natoms=1,
                          orbitals=False)
    rng = np.random.default_rng(9)
    s.kAc0 = rng.uniform(-0.3, 0.3, (3, nk))
    s.occ = rng.uniform(0.1, 2.0, (nk, nb))
    s.zu = rng.standard_normal((nk, nb, s.NL)) + 1j * rng.standard_normal((nk, nb, s.NL))
    print(f"[gpu] density {N} {nk} x {nb}", flush=True)
    with gpu.Context(s, prec) as c:
        rho = c.psi_rho_RT()
        z = np.asarray(c.get_orbitals()).astype(np.complex128)
    ref = np.einsum("kb,kbp->p", s.occ, z.real ** 2 + z.imag ** 2)
    assert np.max(np.abs(rho - ref) / ref) < nk * nb * 1.1e-16
