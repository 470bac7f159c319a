"""The plane transforms (csrc/dft.hpp) on planes of long lines, whose sums neighbouring
lanes share (2, 4 or 8 of them) and whose blocks take one line to eight: the Hartree
solve against numpy's FFT, and the kinetic preconditioner inside the CG against the
oracle.

Tolerances: as for the Hartree solve on other grids, 1e-12 relative to the largest
V_H; the CG's 1e-12.
"""
import math

import numpy as np
import pytest

from helpers import rel
from oracle.cpu import Oracle
from salmon_amd import gpu, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [(8, 8, 256), (8, 256, 8), (10, 200, 200), (9, 65, 97), (8, 129, 64), (20, 20, 256), (8, 256, 256),
                               (40, 33, 70), (12, 12, 100)])
def test_hartree_matches_fft(N):
    s = synth.make_system(N=N, L=tuple(0.64 * n for n in N), nk3=(1, 1, 1), NB=1, seed=2, atoms="random", natoms=1,
                          orbitals=False)
    rho = 0.02 + 0.3 * np.random.default_rng(6).random(s.NL)
    print(f"[gpu] hartree {N}", flush=True)
    with gpu.Context(s, gpu.FP64) as c:
        vh, _ = c.hartree_xc(rho, gpu.XC_NONE)
    g = [2 * math.pi * np.fft.fftfreq(n, 1.0 / n) / a for n, a in zip(N, (s.aLx, s.aLy, s.aLz))]
    g2 = g[0][:, None, None] ** 2 + g[1][None, :, None] ** 2 + g[2][None, None, :] ** 2
    g2[0, 0, 0] = 1.0
    f = 4 * math.pi * np.fft.fftn(rho.reshape(N)) / g2
    f[0, 0, 0] = 0.0
    assert rel(vh, np.fft.ifftn(f).real.reshape(-1)) < 1e-12


@pytest.mark.parametrize("N,nk", [((8, 8, 64), 1), ((8, 64, 9), 3), ((9, 64, 50), 1), ((8, 33, 64), 2)])
def test_kinetic_preconditioner_in_the_cg(N, nk):
    s = synth.make_system(N=N, L=tuple(0.64 * n for n in N), nk3=(nk, 1, 1), NB=2, seed=41, atoms="random", natoms=2,
                          rc=1.7, sigma=0.7)
    print(f"[gpu] kinetic {N} x {nk}", flush=True)
    zr, evr, itr = Oracle(s).cg(s.kAc0, s.zu, 2, precond=gpu.PC_KINETIC)
    with gpu.Context(s, gpu.FP64) as c:
        ev, it = c.cg(s.kAc0, 2, gpu.PC_KINETIC)
        assert rel(c.get_orbitals(), zr) < 1e-12 and rel(ev, evr) < 1e-12 and np.array_equal(it, itr)
