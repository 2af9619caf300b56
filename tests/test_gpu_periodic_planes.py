"""A periodic layer that contains the reflection plane (negative sca_offset):
the monitors hold E after the metal update of the same step, as the step by
separate calls leaves it, bit for bit; planes in front of, on either side of
and inside the layer, and both materials of the local models."""
import numpy as np
import pytest

import fdtd_amd
from conftest import small_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("offset,material", [(-3, 3), (-3, 7), (-2, 3), (-6, 3), (5, 3)])
def test_samples_of_a_plane_in_the_layer(offset, material):
    out = []
    for fused in (True, False):
        p = small_params(fdtd_amd, sphere=0, block=8, nfreq=5)
        p.periodic_xy, p.NcpmlX, p.NcpmlY, p.NcpmlZ = 1, 0, 0, 8
        p.NCELLX, p.NCELLY, p.NCELLZ = 66, 5, 80
        p.tfsf_inset, p.sca_offset, p.material = 10, offset, material
        s = fdtd_amd.Simulation(p)
        k0 = s.info.tfsf[2] + 2
        s.add_layer(k0, k0 + 4)
        (s.step if fused else s.split_step)(300)
        out.append([s.get_field(c) for c in range(6)] + [s.get_dft(f, c) for f in (4, 5) for c in range(4)])
    assert max(np.abs(d).max() for d in out[1][6:10]) > 0   # on the reflection plane
    for a, b in zip(*out):
        assert np.array_equal(a, b)
