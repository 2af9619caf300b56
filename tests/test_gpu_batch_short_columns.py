"""Batches whose short columns (2 waves) take blocks of 4: alone in the batch, and
as most of one beside taller grids; odd rows and planes, with and without metal,
by graph and directly.  Each simulation gives the bits it gives alone."""
import numpy as np
import pytest

import fdtd_amd
from conftest import small_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("graph", [True, False])
@pytest.mark.parametrize("few,tall", [(3, False), (40, True)])
def test_short_columns_equal_each_alone(few, tall, graph):
    def sims():
        shapes = [(24 + q % 5, 21 + q % 4, 24 + q % 7) for q in range(few)] + ([(25, 22, 150), (21, 27, 270)] if tall else [])
        out = []
        for q, n in enumerate(shapes):
            p = small_params(fdtd_amd, sphere=q % 2, radius=6e-9, nfreq=3)
            p.NCELLX, p.NCELLY, p.NCELLZ = n
            s = fdtd_amd.Simulation(p)
            rng = np.random.default_rng(q)
            for c in range(3):
                s.set_field(c, (rng.standard_normal(s.shape) * 0.1).astype(np.float32))
            out.append(s)
        return out
    a, b = sims(), sims()
    batch = fdtd_amd.Batch(a, flags=0 if graph else fdtd_amd.BATCH_NO_GRAPH)
    batch.run(43)
    for s, t in zip(a, b):
        t.step(43)
        for c in range(6):
            assert np.array_equal(s.get_field(c), t.get_field(c)), (s.shape, c)
        for x, y in zip(s.get_line(), t.get_line()):
            assert np.array_equal(x, y)
