"""Injections added by the general transposed kernel itself (over the whole
grid) against the same reverse sweep cut into single steps' segments and into
segments of odd lengths, with the objective cell in a z slab, a corner, beside
the design block and at the grid's centre plane: the same gradient bits."""
import numpy as np
import pytest

import fdtd_amd
from conftest import small_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("at", [(20, 20, 1), (0, 0, 0), (1, 32, 31), (17, 17, 14), (32, 16, 32)])
def test_objective_cells_of_the_general_kernel(at, monkeypatch):
    monkeypatch.setenv("FDTD_ADJ_PATH", "general")
    out = []
    for ckpt in (0, 1, 7):
        p = small_params(fdtd_amd, n=22, ncpml=5, sphere=0)
        s = fdtd_amd.Simulation(p)
        assert s.shape == (33, 33, 33)
        s.set_design((14, 15, 16), np.random.default_rng(2).uniform(0.1, 0.9, size=(4, 3, 2)).astype(np.float32))
        r = np.random.default_rng(1)
        for q in range(3):
            s.set_field(q, (r.standard_normal(s.shape) * 0.1).astype(np.float32))
        J, g = s.adjoint(24, at, [4e14, 5e14], checkpoint=ckpt)
        out.append((J, g))
    # E on the grid's outer planes is not updated, so a cell in its corner passes nothing on
    assert (np.abs(out[0][1]).max() > 0) == (min(at) > 0 and max(at) < 32)
    for J, g in out[1:]:
        assert J == out[0][0] and np.array_equal(g, out[0][1])
