"""Field and checkpoint read-outs through the pinned halves: sizes below the
threaded copy, of one, two and several chunks, with a short last one."""
import threading

import numpy as np
import pytest

import fdtd_amd
from conftest import small_params

pytestmark = pytest.mark.gpu


def sim(n):
    p = small_params(fdtd_amd, sphere=0)
    p.NCELLX, p.NCELLY, p.NCELLZ = n
    return fdtd_amd.Simulation(p)


# bytes of a field: 0.2, 1.0, 1.1, 15.8, 17.1 and 35 MB
@pytest.mark.parametrize("n", [(24, 24, 24), (50, 50, 53), (50, 50, 58), (144, 144, 144), (149, 148, 148), (193, 190, 198)])
def test_fields_come_back_whole(n):
    s = sim(n)
    rng = np.random.default_rng(n[0])
    f = rng.standard_normal(s.shape, dtype=np.float32)
    for c in (0, 4):
        s.set_field(c, f)
        assert np.array_equal(s.get_field(c), f)
    t = sim(n)
    t.restore(s.checkpoint())
    assert np.array_equal(t.get_field(4), f)


def test_read_outs_on_several_threads():
    sims = [sim((60 + 8 * q, 64, 70)) for q in range(4)]
    fields = [np.random.default_rng(q).standard_normal(s.shape, dtype=np.float32) for q, s in enumerate(sims)]
    for s, f in zip(sims, fields):
        s.set_field(2, f)
    bad = []

    def work(s, f):
        for _ in range(5):
            if not np.array_equal(s.get_field(2), f):
                bad.append(s.shape)
    threads = [threading.Thread(target=work, args=a) for a in zip(sims, fields)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
