"""The one-launch steps on columns of 6 to 16 waves, where their row tiles and
block bounds change (two tiles of 6 waves, one of 8, 12 and 16), against the
pieces on streams: the same bits, forward and transposed."""
import numpy as np
import pytest

import fdtd_amd
from conftest import small_params

pytestmark = pytest.mark.gpu


def pair(n, ncpml, monkeypatch):
    p = small_params(fdtd_amd, sphere=0)
    p.NCELLX, p.NCELLY, p.NCELLZ = n
    p.NcpmlX, p.NcpmlY, p.NcpmlZ = ncpml
    p.inc_phi = 90.0
    for one in ("1", "0"):
        monkeypatch.setenv("FDTD_ONE_LAUNCH", one)
        s = fdtd_amd.Simulation(p)
        assert (s.get_info().tile[6] == 0) == (one == "1")
        rng = np.random.default_rng(n[2])
        for c in range(6):
            s.set_field(c, (rng.standard_normal(s.shape) * 0.1).astype(np.float32))
        yield s


@pytest.mark.parametrize("n,ncpml", [((24, 21, 318), (6, 5, 7)), ((21, 24, 420), (5, 6, 6)), ((20, 20, 600), (5, 5, 5)),
                                     ((20, 21, 800), (5, 5, 5))])
def test_forward(n, ncpml, monkeypatch):
    out = []
    for s in pair(n, ncpml, monkeypatch):
        s.step(30)
        out.append([s.get_field(c) for c in range(6)] + [s.flux()["raw"], *s.get_line()])
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("nz", [340, 420])
def test_transposed(nz, monkeypatch):
    rho = np.random.default_rng(nz).uniform(0.1, 0.9, size=(5, 4, 3)).astype(np.float32)
    out = []
    for s in pair((20, 22, nz), (6, 6, 6), monkeypatch):
        c = [e // 2 for e in s.shape]
        lo = [c[0] - 2, c[1] - 2, c[2] - 1]
        s.set_design(lo, rho)
        J, g = s.adjoint(30, (c[0], c[1], lo[2] + 4), [4e14, 5e14], checkpoint=12)
        out.append([np.array(J), g] + [s.get_field(q) for q in range(6)])
    assert np.abs(out[0][1]).max() > 0
    for a, b in zip(*out):
        assert np.array_equal(a, b)
