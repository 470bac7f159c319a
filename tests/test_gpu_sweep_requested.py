"""The persistent sweep asked for by name (SALMON_PATH_SWEEP, SALMON_BATCH_SWEEP) on
grids where the automatic choice takes the LDS-resident kernel: it is the sweep that
runs, and every use of it (runs, ETRS, the self-consistent potential,
re-orthonormalisation, the hamiltonian and observables entries, batches, a change
of path) follows the streamed kernels.  Which of the two the automatic choice takes
around its limits.

Tolerances as in the sweep's other tests: FP64 1e-12 relative, complex64 1e-5.
"""
import numpy as np
import pytest

from helpers import rel
from salmon_amd import gpu, synth
from test_gpu_resident import GRIDS, TOL, cell

pytestmark = pytest.mark.gpu
SWEEP = [(8, 8, 8), (9, 10, 11), (12, 8, 10), (12, 12, 12), (13, 9, 8), (12, 14, 16)]


def run(s, path, prec, n, prop=gpu.PROP_MIDPOINT, scf=False, reortho=0, resident=-1):
    ac = synth.acos2_pulse(n + 1, s.dt, 0.05, 0.3, 4.0)
    with gpu.Context(s, prec) as c:
        c.set_path(path)
        c.set_propagator(prop)
        if scf:
            c.set_scf(s.vloc, gpu.XC_PZ)
        assert c.path() == (gpu.PATH_STREAMED if path == gpu.PATH_STREAMED else gpu.PATH_SWEEP)
        r = c.rt_run(ac, n, reortho_every=reortho)
        assert c.resident() == resident
        r["zu"] = c.get_orbitals()
        k = s.kAc0 + ac[n][:, None]
        c.hamiltonian(k, s.dt)
        r["zu1"] = c.get_orbitals()
        r["J1"], r["E1"], r["n1"] = c.current(k), np.array(c.total_energy(k)), np.array(c.norm())
    return r


def close(a, b, tol):
    for x in a:
        assert rel(a[x], b[x]) < tol, x


@pytest.mark.parametrize("prec", [gpu.FP64, gpu.MIXED])
@pytest.mark.parametrize("N", SWEEP)
def test_sweep_by_name(N, prec):
    s = cell(N)
    close(run(s, gpu.PATH_SWEEP, prec, 3, resident=0), run(s, gpu.PATH_STREAMED, prec, 3), TOL[prec])


@pytest.mark.parametrize("prec", [gpu.FP64, gpu.MIXED])
@pytest.mark.parametrize("prop,scf,reortho", [(gpu.PROP_ETRS, False, 0), (gpu.PROP_ETRS, False, 2), (gpu.PROP_MIDPOINT, True, 2),
                                              (gpu.PROP_ETRS, True, 2), (gpu.PROP_MIDPOINT, False, 2)])
@pytest.mark.parametrize("N", [(9, 10, 11), (12, 8, 10)])
def test_sweep_by_name_step_by_step(N, prop, scf, reortho, prec):
    s = cell(N, natoms=3)
    a = [run(s, path, prec, 4, prop, scf, reortho, res)
         for path, res in ((gpu.PATH_SWEEP, 0), (gpu.PATH_STREAMED, -1))]
    close(*a, TOL[prec])


@pytest.mark.parametrize("prec", [gpu.FP64, gpu.MIXED])
def test_change_between_the_two(prec):
    """The automatic choice, the sweep by name, and back: the plan follows, and the trajectory."""
    s = cell((9, 10, 11))
    ac = synth.acos2_pulse(7, s.dt, 0.05, 0.3, 4.0)
    out = []
    for paths in ((gpu.PATH_AUTO, gpu.PATH_SWEEP, gpu.PATH_AUTO), (gpu.PATH_STREAMED,) * 3):
        with gpu.Context(s, prec) as c:
            J = []
            for i, path in enumerate(paths):
                c.set_path(path)
                J.append(c.rt_run(ac[2 * i:], 2)["J"])
                assert c.resident() == {gpu.PATH_AUTO: 1, gpu.PATH_SWEEP: 0, gpu.PATH_STREAMED: -1}[path]
            out.append(dict(J=np.concatenate(J), zu=c.get_orbitals()))
    close(*out, TOL[prec])


@pytest.mark.parametrize("prec", [gpu.FP64, gpu.MIXED])
@pytest.mark.parametrize("kernel,extra,resident", [
    (gpu.BATCH_SWEEP, None, 0), (gpu.BATCH_AUTO, None, 1), (gpu.BATCH_AUTO, (17, 16, 16), 1), (gpu.BATCH_AUTO, (19, 16, 16), 0),
    (gpu.BATCH_AUTO, (20, 20, 28), 0), (gpu.BATCH_SWEEP, (19, 16, 16), 0), (gpu.BATCH_AUTO, "many", 0)])
def test_batches(kernel, extra, resident, prec):
    """Small odd systems in one batch, alone and beside a grid past the resident kernel's or an orbital count past its
    rounds; per-system fields."""
    systems = [cell((8, 8, 8), nk=1, seed=1), cell((9, 10, 11), seed=2, natoms=3), cell((12, 8, 10), seed=3)]
    if extra == "many":
        systems.append(cell((8, 8, 9), nk=64, nb=20, natoms=1, seed=4))
    elif extra:
        systems.append(cell(extra, nk=1, nb=2, seed=4))
    n = 3
    ac = np.stack([synth.acos2_pulse(n, 0.08, 0.05 / (i + 1), 0.3, 4.0) for i in range(len(systems))])
    ctx = [gpu.Context(s, prec) for s in systems]
    with gpu.Batch(ctx, prec) as b:
        b.set_kernel(kernel)
        assert b.resident() == -1
        r = b.rt_run_ms(ac, n, 0.08)
        assert b.kernel() == gpu.BATCH_SWEEP and b.resident() == resident
    zu = [c.get_orbitals() for c in ctx]
    for i, s in enumerate(systems):
        with gpu.Context(s, prec) as c:
            c.set_path(gpu.PATH_STREAMED)
            q = c.rt_run(ac[i], n, dt=0.08)
            assert rel(zu[i], c.get_orbitals()) < TOL[prec]
        for x in ("J", "E", "norm"):
            assert rel(r[x][i], q[x]) < TOL[prec], (i, x)
    for c in ctx:
        c.close()


@pytest.mark.parametrize("prec", [gpu.FP64, gpu.MIXED])
@pytest.mark.parametrize("N", GRIDS + [(8, 16, 18)])
def test_grids_the_resident_kernel_takes(N, prec):
    """By the automatic choice; (8, 16, 18) has planes of five blocks of 64 columns."""
    s = cell(N)
    a = run(s, gpu.PATH_AUTO, prec, 2, resident=1)
    if N not in GRIDS:
        close(a, run(s, gpu.PATH_STREAMED, prec, 2), TOL[prec])
