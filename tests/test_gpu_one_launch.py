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


@pytest.mark.parametrize("n,ncpml,block,r0", [((20, 22, 24), 5, (5, 4, 3), "clean"), ((26, 20, 40), 6, (4, 6, 5), "x slab"),
                                              ((24, 33, 110), 5, (7, 5, 6), "corner"), ((22, 20, 38), 6, (3, 3, 3), "clean")])
def test_transposed_step_in_one_launch_gives_the_streams_bits(n, ncpml, block, r0, monkeypatch):
    """k_adj_all (and the last grid, whose wave edge lies in the far z slab: the
    general transposed kernel) against the transposed step on streams."""
    p = small_params(fdtd_amd, ncpml=ncpml, sphere=0)
    p.NCELLX, p.NCELLY, p.NCELLZ = n
    p.inc_phi = 90.0
    rng = np.random.default_rng(n[2])
    rho = rng.uniform(0.1, 0.9, size=block).astype(np.float32)
    out = []
    for one in ("1", "0"):
        monkeypatch.setenv("FDTD_ONE_LAUNCH", one)
        s = fdtd_amd.Simulation(p)
        c = [e // 2 for e in s.shape]
        lo = [a - b // 2 for a, b in zip(c, block)]
        s.set_design(lo, rho)
        r = np.random.default_rng(1)
        for q in range(3):
            s.set_field(q, (r.standard_normal(s.shape) * 0.1).astype(np.float32))
        at = {"clean": (c[0], c[1], lo[2] + block[2] + 1), "x slab": (2, c[1], c[2]), "corner": (2, 3, c[2])}[r0]
        J, g = s.adjoint(50, at, [4e14, 5e14], checkpoint=20)
        out.append([np.array(J), g] + [s.get_field(q) for q in range(6)])
    assert np.abs(out[0][1]).max() > 0
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("n", [(24, 24, 24), (33, 21, 70), (90, 70, 64)])
def test_general_kernel_chunks_by_rule(n, monkeypatch):
    """The general kernel with the x chunk its rule takes against chunks of 32 planes."""
    monkeypatch.setenv("FDTD_PATH", "general")
    p = small_params(fdtd_amd)
    p.NCELLX, p.NCELLY, p.NCELLZ = n
    out = []
    for ic in (None, "32"):
        if ic:
            monkeypatch.setenv("FDTD_ICHUNK", ic)
        s = fdtd_amd.Simulation(p)
        assert s.get_info().fused_path == 0
        s.step(200)
        out.append([s.get_field(c) for c in range(6)])
    for c in range(6):
        scale = max(np.abs(f).max() for f in (out[1][:3] if c < 3 else out[1][3:]))
        assert np.abs(out[0][c] - out[1][c]).max() <= 1e-5 * scale, c


@pytest.mark.parametrize("graph", [True, False])
def test_batch_of_every_column_height_equals_each_alone(graph):
    """Grids of 2, 3, 4, 5, 6 and 8 waves a column in one batch: the first five
    share blocks of 12 waves (6, 4, 3, 2 and 2 row tiles, two waves idle at 5),
    the last has blocks of 8.  203 steps, so periods by graph and single steps."""
    def sims():
        out = []
        for q, (nx, ny, nz) in enumerate(((24, 24, 24), (21, 27, 131), (22, 24, 200), (20, 23, 270), (25, 20, 330), (20, 21, 400))):
            p = small_params(fdtd_amd, sphere=q % 2, radius=6e-9)
            p.NCELLX, p.NCELLY, p.NCELLZ = nx, ny, nz
            s = fdtd_amd.Simulation(p)
            rng = np.random.default_rng(q)
            for c in range(3):
                s.set_field(c, (rng.standard_normal(s.shape) * 0.1).astype(np.float32))
            out.append(s)
        return out
    a, b = sims(), sims()
    batch = fdtd_amd.Batch(a, flags=0 if graph else fdtd_amd.BATCH_NO_GRAPH)
    assert all(batch.tile(i)[:2] == (1, 2) for i in range(len(a)))
    batch.run(203)
    for s, t in zip(a, b):
        t.step(203)
        for c in range(6):
            assert np.array_equal(s.get_field(c), t.get_field(c)), (s.shape, c)
        for x, y in zip(s.get_line(), t.get_line()):
            assert np.array_equal(x, y)
