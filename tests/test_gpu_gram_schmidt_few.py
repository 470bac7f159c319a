"""Gram-Schmidt around the band count (4) from which it runs in panels, against the
sequential loop in NumPy; first, second and third calls (eager, captured, replayed
below it).

Tolerance: as for the panels, 1e-12 on random bands, whose angles stay near one.
"""
import numpy as np
import pytest

from helpers import rel
from salmon_amd import gpu, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb", [1, 2, 3, 4, 5])
def test_few_bands_match_the_sequential_loop(nb):
    N, nk = (9, 8, 13), 3
    s = synth.make_system(N=N, L=tuple(0.64 * n for n in N), nk3=(nk, 1, 1), NB=nb, seed=4, atoms="random", natoms=1,
                          orbitals=False)
    rng = np.random.default_rng(4)
    s.zu = rng.standard_normal((nk, nb, s.NL)) + 1j * rng.standard_normal((nk, nb, s.NL))
    ref = s.zu.copy()
    for k in range(nk):
        for b in range(nb):
            for j in range(b):
                ref[k, b] -= ref[k, j] * (np.vdot(ref[k, j], ref[k, b]) * s.Hxyz)
            ref[k, b] /= np.sqrt(np.vdot(ref[k, b], ref[k, b]).real * s.Hxyz)
    with gpu.Context(s, gpu.FP64) as c:
        for call in range(3):
            print(f"[gpu] {nb} bands, call {call}", flush=True)
            c.put_orbitals(s.zu)
            c.gram_schmidt()
            assert rel(c.get_orbitals(), ref) < 1e-12
