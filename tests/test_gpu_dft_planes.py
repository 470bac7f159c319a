"""The Hartree solve's plane transforms (csrc/dft.hpp) against numpy's FFT where
their blocks and tiles end: axes shorter and longer than a block's lines, planes of
several staged tiles, lines longer than a thread block covers twice, the longest
axis (256) in each place, and one x line per block.

Tolerance: six direct sums of up to 256 terms with twiddles and products rounded
to 1.1e-16 each; sqrt(6 * 256) * 1.1e-16 = 4e-15 if they add at random, and the
largest rho(G) is not the largest V(G): 1e-12 relative to the largest V_H, as for
the other grids.
"""
import math

import numpy as np
import pytest

from helpers import rel
from salmon_amd import gpu, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [(8, 8, 8), (9, 33, 8), (8, 9, 70), (17, 40, 41), (8, 8, 256), (8, 256, 9), (256, 8, 9),
                               (129, 8, 8), (8, 200, 130)])
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
    ref = np.fft.ifftn(f).real.reshape(-1)
    print(f"[gpu]   {rel(vh, ref):.2e}", flush=True)
    assert rel(vh, ref) < 1e-12
