"""The CG's exit (|ev - <x|H|x>| < 1e-15, CG.f90:114) on grids whose last block is
partly past the grid: one k point's bands are converged and leave their iterations,
the other's are random and go on; eager, captured and replayed.

Tolerances: the random k point as in the CG's other tests against the oracle,
1e-12, for two iterations; each of the three more multiplies an error by at most the
ratio of successive residuals, a few: 1e-10.  The converged one's orbitals move
within what the exit test resolves, sqrt(1e-15) over the gaps of a few tenths: 1e-6.
"""
import numpy as np
import pytest

from helpers import rel
from oracle.cpu import Oracle
from salmon_amd import gpu, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precond", [gpu.PC_NONE, gpu.PC_KINETIC])
@pytest.mark.parametrize("N", [(9, 9, 9), (9, 10, 11), (8, 8, 9)])
def test_one_k_point_leaves_its_iterations(N, precond):
    nb, ncg = 3, 5
    s = synth.make_system(N=N, L=tuple(0.64 * n for n in N), nk3=(2, 1, 1), NB=nb, seed=43, atoms="random", natoms=3,
                          rc=1.7, sigma=0.7)
    assert s.NL % 256
    print(f"[gpu] cg exit {N} precond {precond}", flush=True)
    with gpu.Context(s, gpu.FP64) as c:
        c.ground_state(s.kAc0, 200, iter_cg_max=ncg, precond=precond, tol=0.0)
        z0 = np.array(c.get_orbitals())
        z0[1] = synth.gram_schmidt(s.zu, s.Hxyz)[1]
        zr, evr, itr = Oracle(s).cg(s.kAc0, z0, ncg, precond=precond)
        out = []
        for call in range(3):
            c.put_orbitals(z0)
            ev, it = c.cg(s.kAc0, ncg, precond)
            z = np.array(c.get_orbitals())
            out.append((z, ev, it))
            it = np.asarray(it).reshape(2, nb)
            print(f"[gpu]   call {call}: iterations {it.tolist()} zu {rel(z[0], zr[0]):.1e} {rel(z[1], zr[1]):.1e}",
                  flush=True)
            assert it[0].max() < ncg and it[1].min() == ncg
            assert rel(z[1], zr[1]) < 1e-10 and rel(z[0], zr[0]) < 1e-6
        for o in out[1:]:
            assert all(np.array_equal(a, b) for a, b in zip(out[0], o))
