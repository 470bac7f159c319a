"""The LDS-resident kernel of the batches and of single contexts off 16^3
(csrc/resident.hpp) against the streamed kernels: every number of x points per
thread it is compiled for, workgroups from one wave to twelve, planes with an
idle tail of lanes, odd axes, overlapping and shared spheres, atoms of fewer
than four projectors and of none, spheres of more than 128 points, runs longer than one
launch's steps; and the systems next to its limits, which the persistent sweep
takes: more projectors per atom, an orbital count past its rounds, a batch with
a larger grid.

Tolerances as in the sweep's own tests: FP64 results differ by the rounding of
sums of a few hundred terms per step, 1e-12 relative; complex64 currents and
energies 1e-5, norms and densities likewise.
"""
import numpy as np
import pytest

from helpers import rel
from salmon_amd import gpu, synth

pytestmark = pytest.mark.gpu
H = 10.26 / 16
TOL = {gpu.FP64: 1e-12, gpu.MIXED: 1e-5}


def cell(N, nk=2, nb=3, natoms=2, seed=5, rc=2.0, h=H):
    s = synth.make_system(N=N, L=tuple(n * h for n in N), nk3=(nk, 1, 1), NB=nb, seed=seed, atoms="random",
                          natoms=natoms, rc=rc)
    return s


def fewer_projectors(s, keep):
    """Keeps the first keep[a] projectors of atom a."""
    sel = [4 * a + l for a, k in enumerate(keep) for l in range(k)]
    s.a_tbl, s.iuV, s.uV = s.a_tbl[sel], s.iuV[sel], np.ascontiguousarray(s.uV[sel])
    return s


def run(s, path, prec, nsteps, ac):
    with gpu.Context(s, prec) as c:
        c.set_path(path)
        r = c.rt_run(ac, nsteps)
        r["zu"] = c.get_orbitals()
        k = s.kAc0 + ac[nsteps][:, None]
        c.hamiltonian(k, s.dt)
        r["zu1"] = c.get_orbitals()
        r["J1"], r["E1"], r["n1"] = c.current(k), np.array(c.total_energy(k)), np.array(c.norm())
    return r


def compare(s, prec, nsteps=3):
    ac = synth.acos2_pulse(nsteps + 1, s.dt, 0.05, 0.3, 4.0)
    a, b = run(s, gpu.PATH_AUTO, prec, nsteps, ac), run(s, gpu.PATH_STREAMED, prec, nsteps, ac)
    for x in a:
        assert rel(a[x], b[x]) < TOL[prec], x


# (y, z) planes of 1 to 6 blocks of 64 columns, x points per thread 1, 2, 3, 4 and 6, odd and short axes, 12 waves full
GRIDS = [(8, 8, 8), (12, 8, 8), (13, 8, 8), (25, 8, 8), (9, 10, 11), (12, 12, 12), (11, 13, 12), (12, 14, 16), (16, 15, 15),
         (8, 16, 24), (31, 8, 9)]


@pytest.mark.parametrize("prec", [gpu.FP64, gpu.MIXED])
@pytest.mark.parametrize("N", GRIDS)
def test_resident_matches_streamed(N, prec):
    compare(cell(N), prec)


@pytest.mark.parametrize("prec", [gpu.FP64, gpu.MIXED])
@pytest.mark.parametrize("case", ["overlap", "few", "none", "large_sphere", "five", "one_atom"])
def test_resident_projector_tables(case, prec):
    if case == "overlap":
        s = cell((8, 9, 10), natoms=6)
    elif case == "few":
        s = fewer_projectors(cell((9, 8, 10), natoms=4), [1, 4, 0, 2])
    elif case == "none":
        s = fewer_projectors(cell((9, 8, 10), natoms=2), [0, 0])
    elif case == "large_sphere":  # more than two passes of 64 points per atom
        s = cell((12, 12, 12), natoms=2, rc=2.6)
        assert s.Mps.max() > 256
    elif case == "five":  # past the kernel's projectors per atom: the sweep
        s = cell((9, 10, 8), natoms=2)
        s.a_tbl = np.array([1] * 5 + [2] * 3, np.int32)
        s.uV = np.where(np.arange(s.Nps)[None, :] < s.Mps[s.a_tbl - 1][:, None], s.uV, 0.0)
    else:
        s = cell((8, 8, 8), natoms=1)
    compare(s, prec)


@pytest.mark.parametrize("prec", [gpu.FP64, gpu.MIXED])
def test_resident_long_run_and_reorthonormalisation(prec):
    """More steps than one launch holds, in one run and in two, and stretches between re-orthonormalisations."""
    s = cell((8, 9, 8), nk=1)
    n = 70
    ac = synth.acos2_pulse(n, s.dt, 0.05, 0.3, 6.0)
    out = []
    for parts, reortho, path in (((n,), 0, gpu.PATH_AUTO), ((33, n - 33), 0, gpu.PATH_AUTO), ((n,), 0, gpu.PATH_STREAMED),
                                 ((n,), 35, gpu.PATH_AUTO), ((n,), 35, gpu.PATH_STREAMED)):
        with gpu.Context(s, prec) as c:
            c.set_path(path)
            r, at = [], 0
            for m in parts:
                r.append(c.rt_run(ac[at:], m, reortho_every=reortho))
                at += m
            out.append(np.concatenate([np.column_stack([x["J"], x["E"], x["norm"]]) for x in r]))
    assert np.array_equal(out[0], out[1])
    assert rel(out[0], out[2]) < TOL[prec] and rel(out[3], out[4]) < TOL[prec]


@pytest.mark.parametrize("prec", [gpu.FP64, gpu.MIXED])
@pytest.mark.parametrize("extra", [None, (17, 16, 16), "many"])
def test_batches_around_the_resident_limits(extra, prec):
    """Small odd systems in one batch: alone (resident, two workgroup shapes), beside a grid that is not resident, and
    with more orbitals than the resident rounds (both on the sweep); per-system fields."""
    systems = [cell((8, 8, 8), nk=1, seed=1), cell((9, 10, 11), seed=2, natoms=3), cell((12, 8, 10), seed=3)]
    if extra == "many":
        systems.append(cell((8, 8, 9), nk=64, nb=20, natoms=1, seed=4))
    elif extra:
        systems.append(cell(extra, nk=1, nb=2, seed=4))
    n = 3
    ac = np.stack([synth.acos2_pulse(n, 0.08, 0.05 / (i + 1), 0.3, 4.0) for i in range(len(systems))])
    ctx = [gpu.Context(s, prec) for s in systems]
    with gpu.Batch(ctx, prec) as b:
        r = b.rt_run_ms(ac, n, 0.08)
        assert b.kernel() == gpu.BATCH_SWEEP
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
