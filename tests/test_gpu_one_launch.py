"""The field update in one launch (k_step_all) against the pieces on streams:
the same cells with the same arithmetic, so the same bits.  Grids from one
plane per chunk to several, odd sizes, uneven CPML, a line of several columns
of waves, with and without metal, and the hydrodynamic box."""
import numpy as np
import pytest

import fdtd_amd
from conftest import small_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,ncpml,sphere,nonlocal_", [((24, 24, 24), (6, 6, 6), 1, 0), ((21, 27, 118), (5, 7, 6), 0, 0),
                                                      ((61, 34, 130), (6, 6, 9), 1, 0), ((131, 70, 190), (9, 6, 8), 1, 0),
                                                      ((24, 25, 26), (6, 5, 6), 1, 3), ((28, 24, 260), (6, 6, 6), 1, 1)])
def test_one_launch_gives_the_streams_bits(n, ncpml, sphere, nonlocal_, monkeypatch):
    p = small_params(fdtd_amd, sphere=sphere)
    p.NCELLX, p.NCELLY, p.NCELLZ = n
    p.NcpmlX, p.NcpmlY, p.NcpmlZ = ncpml
    p.NONLOCAL = nonlocal_
    p.inc_phi = 90.0
    out = []
    for one in ("1", "0"):
        monkeypatch.setenv("FDTD_ONE_LAUNCH", one)
        s = fdtd_amd.Simulation(p)
        assert s.get_info().fused_path == 1
        assert (s.get_info().tile[6] == 0) == (one == "1")
        rng = np.random.default_rng(n[2])
        for c in range(6):
            s.set_field(c, (rng.standard_normal(s.shape) * 0.1).astype(np.float32))
        s.step(41)
        s.step(30)
        out.append([s.get_field(c) for c in range(6)] + [s.flux()["raw"], *s.get_line()])
    for a, b in zip(*out):
        assert np.array_equal(a, b)
