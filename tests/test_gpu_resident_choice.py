"""Which kernel the automatic choice takes on grids that fit the LDS-resident one:
that one for few orbitals and wherever it was measured faster, the sweep for many
orbitals of grids that leave its threads idle (14^3: 196 of 256 columns, six x points
per thread).  Both follow the streamed kernels.

Tolerances as in the sweep's other tests: FP64 1e-12 relative, complex64 1e-5.
"""
import numpy as np
import pytest

from helpers import rel
from salmon_amd import gpu, synth
from test_gpu_resident import TOL, cell

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,nk,nb,natoms,prec,resident", [
    ((14, 14, 14), 2, 4, 1, gpu.FP64, 1), ((14, 14, 14), 16, 16, 1, gpu.FP64, 1), ((14, 14, 14), 32, 32, 1, gpu.FP64, 0),
    ((14, 14, 14), 2, 4, 1, gpu.MIXED, 1), ((14, 14, 14), 25, 31, 1, gpu.MIXED, 0), ((31, 8, 9), 32, 32, 1, gpu.FP64, 0),
    ((31, 8, 9), 2, 3, 1, gpu.FP64, 1), ((12, 12, 12), 32, 32, 1, gpu.FP64, 1), ((8, 8, 8), 32, 32, 1, gpu.MIXED, 1),
    ((12, 12, 12), 32, 32, 6, gpu.FP64, 1)])
def test_choice(N, nk, nb, natoms, prec, resident):
    s = cell(N, nk=1, nb=1, natoms=natoms)
    rng = np.random.default_rng(5)
    s.kAc0 = rng.uniform(-0.3, 0.3, (3, nk))
    s.occ = np.full((nk, nb), 2.0 / nk)
    s.zu = (rng.standard_normal((nk, nb, s.NL)) + 1j * rng.standard_normal((nk, nb, s.NL))) / np.sqrt(2 * s.NL * s.Hxyz)
    ac = synth.acos2_pulse(4, s.dt, 0.05, 0.3, 4.0)
    out = []
    for path in (gpu.PATH_AUTO, gpu.PATH_STREAMED):
        with gpu.Context(s, prec) as c:
            c.set_path(path)
            r = c.rt_run(ac, 3)
            assert c.resident() == (resident if path == gpu.PATH_AUTO else -1)
            r["zu"] = c.get_orbitals()
            out.append(r)
    for x in out[0]:
        assert rel(out[0][x], out[1][x]) < TOL[prec], x


@pytest.mark.parametrize("prec", [gpu.FP64, gpu.MIXED])
@pytest.mark.parametrize("grids,resident", [
    ([(8, 8, 8), (8, 9, 10), (9, 10, 11), (10, 10, 10), (11, 11, 11), (12, 12, 12), (12, 10, 8), (13, 13, 13), (14, 14, 14),
      (15, 15, 15), (8, 16, 16), (16, 8, 16), (16, 12, 12), (24, 8, 8), (31, 8, 9), (10, 12, 14)], 0),
    ([(8, 8, 8), (12, 12, 12), (16, 16, 16)], 1)])
def test_choice_for_batches_of_shapes(grids, resident, prec):
    """Many shapes would be as many launches of the resident kernel, one after another; few are not too many."""
    systems = [cell(N, nk=2, nb=2, natoms=2, seed=i) for i, N in enumerate(grids)]
    ac = synth.acos2_pulse(3, 0.08, 0.05, 0.3, 4.0)
    ctx = [gpu.Context(s, prec) for s in systems]
    with gpu.Batch(ctx, prec) as b:
        r = b.rt_run(ac, 2, 0.08)
        assert b.resident() == resident
    for i, s in enumerate(systems):
        ctx[i].close()
        with gpu.Context(s, prec) as c:
            c.set_path(gpu.PATH_STREAMED)
            q = c.rt_run(ac, 2, dt=0.08)
        for x in ("J", "E", "norm"):
            assert rel(r[x][i], q[x]) < TOL[prec], (i, x)
