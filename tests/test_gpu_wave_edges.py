"""Grids whose far z slab starts at, just before and just after the edge of a
wave of the row-blocked kernel (waves without z-slab lanes run a march without
the z-CPML work), and columns of two to four waves, against the split path."""
import numpy as np
import pytest

import fdtd_amd
from conftest import small_params

pytestmark = pytest.mark.gpu


# the middle wave of three holds k = 63 .. 126; the far slab starts at NZ - 1 - 6
@pytest.mark.parametrize("nz,first_far", [(119, 125), (120, 126), (121, 127), (176, 182), (184, 190), (50, 56)])
def test_far_slab_at_a_wave_edge(nz, first_far):
    p = small_params(fdtd_amd, n=20, sphere=0)
    p.NCELLZ = nz
    fields = []
    for split in (False, True):
        s = fdtd_amd.Simulation(p)
        assert s.shape[2] - 1 - 6 == first_far
        assert s.get_info().fused_path == 1
        rng = np.random.default_rng(nz)
        for c in range(3):
            s.set_field(c, (rng.standard_normal(s.shape) * 0.1).astype(np.float32))
        (s.split_step if split else s.step)(60)
        fields.append([s.get_field(c) for c in range(6)])
    for c in range(6):
        scale = max(np.abs(f).max() for f in fields[1][:3] if c < 3) if c < 3 else max(np.abs(f).max() for f in fields[1][3:])
        # both are FP32; they differ in where the plane wave's terms are added
        assert np.abs(fields[0][c] - fields[1][c]).max() <= 1e-5 * scale, c
