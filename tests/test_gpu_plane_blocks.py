"""Whole-grid kernels whose blocks take 256 consecutive cells of a y-z plane
(split path, periodic mode): planes of a multiple of 256 cells, one row more
and odd sizes; the split TFSF kernel on its plane cells; periodic wraps on the
narrowest grids.  Against the fused step, and against the oracle."""
import numpy as np
import pytest

import fdtd_amd
import oracle as O
from conftest import small_params

pytestmark = pytest.mark.gpu


def errors(a, b):
    me = max(np.abs(f).max() for f in b[:3])
    mh = max(np.abs(f).max() for f in b[3:])
    return max(float(np.abs(x - y).max() / (me if c < 3 else mh)) for c, (x, y) in enumerate(zip(a, b)))


@pytest.mark.parametrize("n,theta", [((20, 19, 51), 0.0), ((21, 20, 51), 30.0), ((22, 23, 29), 90.0)])
def test_split_path_on_odd_planes(n, theta):
    p = small_params(fdtd_amd, sphere=0)
    p.NCELLX, p.NCELLY, p.NCELLZ = n
    p.inc_theta = theta
    p.inc_phi = 40.0
    s, f = fdtd_amd.Simulation(p), fdtd_amd.Simulation(p)
    s.split_step(220)
    f.step(220)
    assert errors([s.get_field(c) for c in range(6)], [f.get_field(c) for c in range(6)]) < 1e-5


@pytest.mark.parametrize("nx,ny,layer", [(4, 4, 3), (5, 16, 0), (7, 8, 4), (16, 5, 2)])
def test_periodic_wraps_on_narrow_grids(nx, ny, layer):
    p = small_params(O, sphere=0)
    p.NCELLX, p.NCELLY, p.NCELLZ = nx, ny, 51
    p.periodic_xy = 1
    p.NcpmlX = p.NcpmlY = 0
    o, s, t = O.Oracle(p), fdtd_amd.Simulation(p), fdtd_amd.Simulation(p)
    rng = np.random.default_rng(nx)
    k0 = s.shape[2] // 2
    for g in (o, s, t):
        if layer:
            g.add_layer(k0, k0 + layer)
    for c in range(3):
        f = (rng.standard_normal(s.shape) * 0.1).astype(np.float32)
        o.set_field(c, f.astype(np.float64))
        s.set_field(c, f)
        t.set_field(c, f)
    o.step(120)
    s.step(120)
    t.split_step(120)
    want = [o.get_field(c) for c in range(6)]
    # 120 FP32 steps against FP64: the bar of the parity tests
    assert errors([s.get_field(c) for c in range(6)], want) < 2e-4
    assert errors([t.get_field(c) for c in range(6)], want) < 2e-4
    a, b = s.reflectance(), o.reflectance()
    assert np.abs(a["T"] - b["T"]).max() <= 1e-4 * np.abs(b["T"]).max()


@pytest.mark.parametrize("nz,steps,stride", [(51, 200, 4), (53, 201, 4), (85, 330, 3), (64, 257, 1)])
def test_incident_power_of_the_replayed_line(nz, steps, stride):
    """R and ref_r share the reflected flux, so their ratio gives the incident
    power at the source plane; a numpy run of the line gives it too.  FP64 on
    both sides and some hundred terms: 1e-10."""
    p = small_params(fdtd_amd, sphere=0)
    p.NCELLX = p.NCELLY = 6
    p.NCELLZ = nz
    p.periodic_xy = 1
    p.NcpmlX = p.NcpmlY = 0
    p.dft_stride = stride
    s = fdtd_amd.Simulation(p)
    rng = np.random.default_rng(nz)
    for c in range(6):
        s.set_field(c, (rng.standard_normal(s.shape) * 0.1).astype(np.float32))
    s.step(steps)
    r = s.reflectance()
    freq, einc = s.spectrum_setup()
    area = 36 * p.dx ** 2
    got = r["ref_r"] * area * np.abs(einc) ** 2 / r["R"]
    i, L, d, dt = s.info, 6 * nz, p.dx, s.info.dt
    c0, ep0, mu0, z0 = 2.99792458e8, 8.85418782e-12, 1.25663706e-6, 376.730313462
    e, h, mur, acc = np.zeros(L), np.zeros(L), [0.0, 0.0], np.zeros(len(freq), complex)
    mc = (c0 * dt - d) / (c0 * dt + d)
    for t in range(steps):
        h[:-1] -= z0 * dt / (mu0 * d) * (e[1:] - e[:-1])
        n = e.copy()
        n[1:-1] -= dt / (z0 * ep0 * d) * (h[1:-1] - h[:-2])
        n[0], n[-1] = mur[0] + mc * (n[1] - e[0]), mur[1] + mc * (n[-2] - e[-1])
        mur = [n[1], n[-2]]
        b = np.float32((t - i.delay) / i.width)
        n[i.m0 - 50] += np.exp(-float(b * b) / 2) * np.sin(2 * np.pi * i.f_0 * dt * t)
        e = n
        if t % stride == 0:
            acc += e[i.m0] * np.exp(2j * np.pi * freq * (t + 1.0) * dt)
    want = np.abs(acc) ** 2 * area
    assert want.min() > 0
    assert np.abs(got / want - 1).max() < 1e-10
