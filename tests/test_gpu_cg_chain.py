"""The band-by-band CG's launches (csrc/cg.hpp) against the oracle where their
blocks and passes end: grids that are no multiple of a block's 64, 256 or 512
points, one band (no lower bands), band counts around the projections' groups
of 8 and passes of 64, and atoms with more projectors than a pass of 16, with
none, and of overlapping spheres.

Tolerance: 1e-12 relative for up to 6 bands, as for the CG's other tests against
the oracle (summation order, grown over the iterations); each band starts from
the projections on all lower ones and inherits their errors, so in proportion
for more.
"""
import numpy as np
import pytest

from helpers import rel
from oracle.cpu import Oracle
from salmon_amd import gpu, synth

pytestmark = pytest.mark.gpu


def uneven_projectors(s):
    """Atom 1 with 18 projectors, atom 2 with none, the others with their four."""
    keep = [l for l in range(s.Nlma) if s.a_tbl[l] != 2]
    first = [l for l in keep if s.a_tbl[l] == 1]
    order = first + [first[i % 4] for i in range(14)] + [l for l in keep if s.a_tbl[l] != 1]
    scale = np.array([1.0 if i < 4 or i >= 18 else 0.2 + 0.02 * i for i in range(len(order))])
    s.a_tbl = np.ascontiguousarray(s.a_tbl[order])
    s.uV = np.ascontiguousarray(s.uV[order] * scale[:, None])
    s.iuV = np.ascontiguousarray(s.iuV[order])
    return s


@pytest.mark.parametrize("precond", [gpu.PC_NONE, gpu.PC_KINETIC])
@pytest.mark.parametrize("N,nk,nb,uneven", [((8, 8, 8), 2, 1, False), ((9, 9, 9), 1, 9, True), ((9, 10, 11), 3, 8, False),
                                            ((13, 8, 21), 1, 17, True), ((8, 8, 8), 1, 66, False)])
def test_cg_at_block_edges(N, nk, nb, uneven, precond):
    s = synth.make_system(N=N, L=tuple(0.64 * n for n in N), nk3=(nk, 1, 1), NB=nb, seed=41, atoms="random", natoms=4,
                          rc=1.7, sigma=0.7, name="edges")
    if uneven:
        s = uneven_projectors(s)
    print(f"[gpu] cg {N} nk {nk} nb {nb} uneven {uneven} precond {precond}", flush=True)
    zr, evr, itr = Oracle(s).cg(s.kAc0, s.zu, 2, precond=precond)
    with gpu.Context(s, gpu.FP64) as c:
        for call in range(3):  # eager, captured, replayed
            c.put_orbitals(s.zu)
            ev, it = c.cg(s.kAc0, 2, precond)
            z = c.get_orbitals()
            tol = 1e-12 * max(1.0, nb / 6)
            print(f"[gpu]   call {call}: zu {rel(z, zr):.2e} esp_var {rel(ev, evr):.2e}", flush=True)
            assert rel(z, zr) < tol
            assert rel(ev, evr) < tol
            assert np.array_equal(it, itr)
