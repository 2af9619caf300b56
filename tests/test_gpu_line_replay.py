"""The incident spectrum that fdtd_reflectance divides by, with the source of the
1D line off its usual cell: beside the source plane, next to either end and on
the last cell.  R and the reference's column share the flux through the
reflection plane, so their quotient is the incident power over the source's: the
line alone, FP64 recurrences of up to 3900 steps on both sides (some 1e-13 of each
other per rounding; 1e-9 of the oracle's value allowed).  The line has 6 NCELLZ
cells: 240 are replayed on the host, 804 (the shortest) and 1800 on the device,
whose staging buffer the steps fit here."""
import numpy as np
import pytest

import fdtd_amd
import oracle as O
from conftest import small_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nz,steps", [(40, 900), (134, 2000), (300, 3900)])
@pytest.mark.parametrize("src", ["m0 - 1", "1", "2", "L - 3", "L - 2", "L - 1"])
def test_incident_power_with_the_source_anywhere_on_the_line(src, nz, steps):
    def params(mod):
        p = small_params(mod, sphere=0, nfreq=4)
        p.periodic_xy, p.NcpmlX, p.NcpmlY, p.NcpmlZ = 1, 0, 0, 8
        p.NCELLX, p.NCELLY, p.NCELLZ = 12, 9, nz
        p.tfsf_inset, p.Tend, p.inc_phi = 10, steps, 90.0
        line = 6 * p.NCELLZ
        p.source_offset = line // 2 - eval(src, {"L": line, "m0": line // 2})
        return p
    s, o = fdtd_amd.Simulation(params(fdtd_amd)), O.Oracle(params(O))
    k0 = s.info.tfsf[2] + 6
    power = []
    for x in (s, o):
        x.add_layer(k0, k0 + 3)
        x.step(steps)
        r = x.reflectance()
        power.append(r["ref_r"] / r["R"])
    print(src, *power, flush=True)
    assert np.abs(power[1]).min() > 0
    assert np.abs(power[0] / power[1] - 1).max() <= 1e-9
