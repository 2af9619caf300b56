"""The TFSF planes of flat and long boxes, whose launches go through each axis's
own rows: fields of the one-launch step, the streams and the separate calls
against the FP64 oracle (2e-4 of the largest value, as the other parity tests),
along every axis and with an oblique wave, whose terms differ on every plane."""
import numpy as np
import pytest

import fdtd_amd
import oracle as O
from conftest import small_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(24, 26, 24), (150, 24, 22), (24, 150, 22), (22, 24, 150), (77, 80, 20), (20, 77, 80), (80, 20, 79)])
def test_planes_of_uneven_boxes(n, monkeypatch):
    def params(mod):
        p = small_params(mod, steps=220, sphere=0)
        p.NCELLX, p.NCELLY, p.NCELLZ = n
        # the incident line has 6 NCELLZ cells: an oblique wave where it is long enough for the box
        if max(n[:2]) <= 2 * n[2]:
            p.inc_theta, p.inc_phi, p.polar_psi = 35.0, 25.0, 40.0
        else:
            p.inc_phi = 90.0
        return p
    o = O.Oracle(params(O))
    o.step(220)
    want = [o.get_field(c) for c in range(6)]
    scale = [max(np.abs(f).max() for f in want[g]) for g in (slice(0, 3), slice(3, 6))]
    assert min(scale) > 0
    for env, split in (({}, False), ({"FDTD_ONE_LAUNCH": "0"}, False), ({}, True)):
        with monkeypatch.context() as m:
            for k, v in env.items():
                m.setenv(k, v)
            s = fdtd_amd.Simulation(params(fdtd_amd))
        (s.split_step if split else s.step)(220)
        err = [float(np.abs(s.get_field(c) - want[c]).max() / scale[c // 3]) for c in range(6)]
        print(n, env, split, ["%.1e" % e for e in err], flush=True)
        assert max(err) < 2e-4
