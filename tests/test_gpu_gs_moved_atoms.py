"""Ground-state state that does not depend on the projector tables stays when an atom
moves and the number of sphere points changes: samples recorded for the learned
preconditioner, and its targets; the CG follows the new tables.

Tolerance: the CG against the oracle, 1e-12 as in its other tests.
"""
import numpy as np
import pytest

from helpers import rel
from oracle.cpu import Oracle
from salmon_amd import gpu, synth
from test_gpu_gs import _moved_atoms

pytestmark = pytest.mark.gpu


def test_samples_and_targets_stay_when_atoms_move():
    s = synth.make_system(N=(12, 12, 12), L=7.0, nk3=(1, 1, 1), NB=4, seed=31, atoms="random", natoms=5)
    t = _moved_atoms(s, (0.41, -0.23, 0.17), 7)
    assert t.Mps.sum() != s.Mps.sum() and t.Nlma == s.Nlma
    print("[gpu] samples across moved atoms", flush=True)
    with gpu.Context(s, gpu.FP64) as c:
        c.pc_record(64, 1)
        c.put_orbitals(s.zu)
        c.cg(s.kAc0, 3, gpu.PC_KINETIC)
        c.pc_set_targets(s.kAc0)
        n, _ = c.pc_samples()
        g = c.pc_get_sample(2)
        assert n == 12
        c.set_projectors(t)
        c.gram_schmidt()
        c.put_orbitals(s.zu)
        ev, it = c.cg(t.kAc0, 2, gpu.PC_KINETIC)
        assert c.pc_samples()[0] == n + 8
        again = c.pc_get_sample(2)
        assert all(np.array_equal(g[x], again[x]) for x in g)
        net = gpu.PcNet(seed=1)
        loss, grad = net.gradient(c, [0, 1])  # (needs the targets)
        assert np.isfinite(loss) and np.all(np.isfinite(grad))
        zr, evr, itr = Oracle(t).cg(t.kAc0, s.zu, 2, precond=gpu.PC_KINETIC)
        assert rel(c.get_orbitals(), zr) < 1e-12 and rel(ev, evr) < 1e-12 and np.array_equal(it, itr)
