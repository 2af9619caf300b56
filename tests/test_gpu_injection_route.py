"""The injection that the general transposed kernel adds itself against one by a
launch of its own (FDTD_ADJ_FUSE_INJECT=0): the same gradient bits, with the
objective cell in every z slab and corner, at the edges of the kernel's tiles
and x chunks, beside the design block and inside it."""
import numpy as np
import pytest

import fdtd_amd
from conftest import small_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ichunk", [None, "3"])
@pytest.mark.parametrize("at,steps", [((20, 20, 1), 40), ((20, 19, 31), 40), ((1, 1, 1), 40), ((31, 31, 31), 40), ((1, 1, 1), 90),
                                      ((31, 31, 31), 90), ((2, 6, 16), 40), ((3, 7, 16), 40), ((5, 8, 17), 40), ((17, 17, 14), 40),
                                      ((15, 16, 16), 40), ((32, 16, 32), 40), ((16, 13, 16), 40)])
def test_injection_in_the_kernel_and_by_its_own_launch(at, steps, ichunk, monkeypatch):
    monkeypatch.setenv("FDTD_ADJ_PATH", "general")
    if ichunk:
        monkeypatch.setenv("FDTD_ICHUNK", ichunk)
    out = []
    for fuse in ("1", "0"):
        monkeypatch.setenv("FDTD_ADJ_FUSE_INJECT", fuse)
        s = fdtd_amd.Simulation(small_params(fdtd_amd, n=22, ncpml=5, sphere=0))
        assert s.shape == (33, 33, 33)
        s.set_design((14, 15, 16), np.random.default_rng(2).uniform(0.1, 0.9, size=(4, 3, 2)).astype(np.float32))
        r = np.random.default_rng(1)
        for q in range(3):
            s.set_field(q, (r.standard_normal(s.shape) * 0.1).astype(np.float32))
        out.append(s.adjoint(steps, at, [4e14, 5e14], checkpoint=16))
    # E on the grid's outer planes is not updated, so a cell there passes nothing on; and the
    # corner cells are 42 cells along the axes from the block, one a step
    away = sum(max(lo - a, a - hi, 0) for a, lo, hi in zip(at, (14, 15, 16), (17, 17, 17)))
    assert (np.abs(out[1][1]).max() > 0) == (min(at) > 0 and max(at) < 32 and away < steps)
    assert out[0][0] == out[1][0] and np.array_equal(out[0][1], out[1][1])


def test_injection_across_two_columns_of_waves(monkeypatch):
    """A grid of two waves a column (62 own cells each), the objective on either side of their edge."""
    monkeypatch.setenv("FDTD_ADJ_PATH", "general")
    for at in ((14, 15, 61), (14, 15, 62), (14, 15, 80)):
        out = []
        for fuse in ("1", "0"):
            monkeypatch.setenv("FDTD_ADJ_FUSE_INJECT", fuse)
            p = small_params(fdtd_amd, ncpml=5, sphere=0)
            p.NCELLX, p.NCELLY, p.NCELLZ = 20, 21, 90
            s = fdtd_amd.Simulation(p)
            s.set_design((14, 15, 64), np.random.default_rng(2).uniform(0.1, 0.9, size=(3, 3, 4)).astype(np.float32))
            r = np.random.default_rng(1)
            for q in range(3):
                s.set_field(q, (r.standard_normal(s.shape) * 0.1).astype(np.float32))
            out.append(s.adjoint(40, at, [4e14, 5e14], checkpoint=0))
        assert np.abs(out[1][1]).max() > 0
        assert out[0][0] == out[1][0] and np.array_equal(out[0][1], out[1][1])
