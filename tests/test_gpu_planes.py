"""Planes of a field read through fdtd_get_slice, against the full-field copy:
the gather kernel packs 256 values of a plane row per block, so rows one
short of it, at it and past it are the sizes to get wrong."""
import numpy as np
import pytest

import fdtd_amd
from conftest import small_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ny,nz", [(18, 242), (242, 24), (30, 243), (243, 22), (24, 241)])
def test_planes_equal_the_field(ny, nz):
    p = small_params(fdtd_amd, sphere=0)
    p.NCELLX, p.NCELLY, p.NCELLZ = 20, ny, nz
    s = fdtd_amd.Simulation(p)
    rng = np.random.default_rng(ny)
    for c in (0, 5):
        f = rng.standard_normal(s.shape).astype(np.float32)
        s.set_field(c, f)
        for axis in range(3):
            for index in (0, s.shape[axis] // 2, s.shape[axis] - 1):
                assert np.array_equal(s.get_slice(c, axis, index), np.take(f, index, axis)), (c, axis, index)
