"""A flat grid with 31 CPML layers, whose psi arrays together pass 4 GB while
every field and every single array stays below: the row-blocked launches reach
each array through a window of its own.  Against the general kernel on planes
in the slabs of all axes, their corners and the interior (1e-5 of the largest
value, the bound of the other comparisons of the two kernels), from fields that
fill the whole grid."""
import numpy as np
import pytest

import fdtd_amd
from conftest import small_params

pytestmark = pytest.mark.gpu


def test_launches_per_variant_with_more_than_4_gb_of_psi(monkeypatch):
    out = []
    for path in ("rows", "general"):
        if path == "general":
            monkeypatch.setenv("FDTD_PATH", "general")
        p = small_params(fdtd_amd, sphere=0, nfreq=1, ncpml=31)
        p.NCELLX = p.NCELLY = 1577
        s = fdtd_amd.Simulation(p)
        nx, ny, nz = s.shape
        assert s.info.fused_path == (path == "rows")
        f = np.random.default_rng(3).random(s.shape, dtype=np.float32)
        f -= 0.5
        for c in range(6):
            s.set_field(c, f if c < 3 else f[:, ::-1])
        del f
        print(path, "set", flush=True)
        s.step(6)
        planes = [(0, 1), (0, 16), (0, nx // 2), (0, nx - 2), (1, 1), (1, 29), (1, ny // 2 + 1), (1, ny - 12), (2, 2), (2, 31), (2, nz // 2),
                  (2, nz - 31), (2, nz - 3)]
        out.append([[s.get_slice(c, a, q) for a, q in planes] for c in range(6)])
        print(path, "read", flush=True)
        s.close()
    for c in range(6):
        scale = max(np.abs(x).max() for k in (range(3) if c < 3 else range(3, 6)) for x in out[1][k])
        for a, b in zip(out[0][c], out[1][c]):
            assert np.abs(b).max() > 0 and np.abs(a - b).max() <= 1e-5 * scale, c
