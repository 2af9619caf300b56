"""The split-BF16 contraction where its sizes end: blocks filled to one slot, to
whole k-steps and past one (the k-steps past the used slots are not run), rows
that do not fill an m-tile, several groups of m-tiles; against the FP64
contraction of the same samples.

Two parts hold 16 bits and a rounding (2^-17 of each operand), lo * lo is left
out (2^-18 at most); three parts are exact to 2^-25 and leave out 3 * 2^-27.
The K products of 3 or 6 terms add in FP32.  Per sample that is at most
2^-15 |x| with two parts, (2^-23 + 6 K 2^-24) |x| with three."""
import numpy as np
import pytest

import fdtd_amd
from conftest import small_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nfreq,block,steps", [(1, 8, 1), (8, 16, 15), (16, 16, 16), (17, 40, 17), (24, 40, 55), (70, 33, 34)])
@pytest.mark.parametrize("mode", [0, 2])
def test_contraction_of_a_partly_filled_block(mode, nfreq, block, steps):
    sims = []
    for exact in (mode, 1):
        p = small_params(fdtd_amd, n=20, ncpml=5, sphere=0, nfreq=nfreq, block=block, exact=exact)
        p.dft_stride = 1
        s = fdtd_amd.Simulation(p)
        rng = np.random.default_rng(3)
        for c in range(6):
            s.set_field(c, (rng.standard_normal(s.shape) * (1.0 if c < 3 else 2.6e-3)).astype(np.float32))
        sims.append(s)
    a, b = sims
    most = np.zeros(6)
    for _ in range(steps):
        a.step(1)
        b.step(1)
        most = np.maximum(most, [np.abs(b.get_field(c)).max() for c in range(6)])
    per_sample = 2.0 ** -15 if mode == 0 else 2.0 ** -23 + 6 * block * 2.0 ** -24
    for face in range(12):
        for comp in range(4):
            x, y = a.get_dft(face, comp), b.get_dft(face, comp)
            tol = per_sample * steps * most[:3].max() if comp < 2 else per_sample * steps * most[3:].max()
            assert np.abs(y).max() > 0
            assert max(np.abs((x - y).real).max(), np.abs((x - y).imag).max()) <= tol, (face, comp)
