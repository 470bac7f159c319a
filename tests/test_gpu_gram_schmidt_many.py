"""Gram-Schmidt of more bands than the CG takes (1024): in panels, and in the
band-by-band form that nearly dependent bands are left to.

Tolerances: random bands in 1.7 times as many dimensions keep a sine of 0.6 or more
to all others, so rounding of 1e-15 grows by the bands' number: 1e-12.  The pair at
a sine of 1e-5: 1e-12 / 1e-5 over the angle.
"""
import numpy as np
import pytest

from helpers import rel
from salmon_amd import gpu, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dependent", [False, True])
def test_more_than_1024_bands(dependent):
    N, nb = (12, 12, 12), 1030
    s = synth.make_system(N=N, L=7.5, nk3=(1, 1, 1), NB=nb, seed=2, atoms="random", natoms=1, orbitals=False)
    rng = np.random.default_rng(2)
    s.zu = rng.standard_normal((1, nb, s.NL)) + 1j * rng.standard_normal((1, nb, s.NL))
    if dependent:
        s.zu[0, 9] = s.zu[0, 3] * (0.7 - 0.4j) + 1e-5 * s.zu[0, 9]
    q, r = np.linalg.qr(s.zu[0].T)
    d = np.diagonal(r)
    ref = (q * (d / np.abs(d))).T / np.sqrt(s.Hxyz)
    with gpu.Context(s, gpu.FP64) as c:
        c.gram_schmidt()
        z = c.get_orbitals()[0]
    o = (z.conj() @ z.T) * s.Hxyz
    assert np.abs(o - np.eye(nb)).max() < 1e-12
    assert rel(z, ref) < (1e-7 if dependent else 1e-12)
