"""The launches per variant and their streams on small grids, which run one
launch a step by default: FDTD_ONE_LAUNCH=0 selects the schedule that grids
above 50 M cells (and batches that hold one, or a simulation without the row
path) take with its defaults.

* fdtd_step: three side streams, the next step's slabs from the join on, the line
  first on the corner stream, the sample with the post-update launch where it
  may: the bits of one stream, and of one launch.
* Batches: direct launches, graph replay, each simulation alone, and a batch that
  mixes row-path and general simulations: the same bits.  Tuned tiles and three
  rows per thread change only rounding (1e-5, as the other tile tests)."""
import numpy as np
import pytest

import fdtd_amd as G
from conftest import small_params
from test_gpu_batch import CASES, build, fields, sims_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hydro,radius,offsets,schedule", [(0, 8e-9, (2, 2), 3), (0, 4e-9, (3, 1), 7),
                                                           (1, 8e-9, (2, 2), 3), (1, 4e-9, (3, 1), 7)])
def test_default_streams_one_stream_and_one_launch(hydro, radius, offsets, schedule, monkeypatch):
    p = small_params(G, steps=300, block=8, radius=radius)
    p.sca_offset, p.abs_offset = offsets
    if hydro:
        p.NONLOCAL = 3
        p.hydro_beta = 1.27e6
    runs = []
    for env, streams, one in (({"FDTD_ONE_LAUNCH": "0"}, 3, False), ({"FDTD_CONCURRENT": "0"}, 0, False), ({}, 0, True)):
        with monkeypatch.context() as m:
            for k, v in env.items():
                m.setenv(k, v)
            s = G.Simulation(p)
            info = s.get_info()
            assert info.tile[6] == streams and (info.tile[5] == 0) == one
            if streams:
                assert info.schedule == schedule | 8
            s.set_point_monitor((9, 8, 7), 300)
            s.step(171)
            s.step(129)
            runs.append(fields(s) + [s.get_dft(f, c) for f in range(12) for c in range(4)] + [*s.point_spectrum([5e14, 6e14])])
    assert np.abs(runs[0][0]).max() > 0 and np.abs(runs[0][-1]).max() > 0
    for other in runs[1:]:
        for a, b in zip(runs[0], other):
            assert np.array_equal(a, b)


def test_batch_on_its_default_streams(monkeypatch):
    steps = 203
    a, b, c = sims_for(CASES), sims_for(CASES), sims_for(CASES)
    monkeypatch.setenv("FDTD_ONE_LAUNCH", "0")
    ba = G.Batch(a, flags=G.BATCH_NO_TUNE)
    bb = G.Batch(b, flags=G.BATCH_NO_TUNE | G.BATCH_NO_GRAPH)
    assert all(ba.tile(i)[2] >= 16 for i in range(len(CASES)))     # not the chunk of one launch (at most 8)
    ba.run(steps)
    bb.run(steps)
    for x, y, z in zip(a, b, c):
        z.step(steps)
        for k, (fa, fb, fc) in enumerate(zip(fields(x), fields(y), fields(z))):
            assert np.array_equal(fa, fb) and np.array_equal(fa, fc), k
        assert np.max(np.abs(x.flux()["raw"] - z.flux()["raw"])) <= 1e-12 * np.max(np.abs(z.flux()["raw"]))


@pytest.mark.parametrize("flags", [G.BATCH_NO_TUNE, G.BATCH_NO_TUNE | G.BATCH_NO_GRAPH])
def test_batch_of_row_path_and_general_simulations(flags, monkeypatch):
    """One simulation without the row path puts the whole batch on the launches per variant."""
    def sims():
        out = sims_for(CASES[:2])
        out += sims_for(CASES[2:3], env_general=True)
        return out + sims_for(CASES[3:])
    a, c = sims(), sims()
    batch = G.Batch(a, flags=flags)
    assert [batch.tile(i)[0] for i in range(4)] == [1, 1, 0, 1] and batch.tile(0)[2] >= 16
    batch.run(203)
    for x, z in zip(a, c):
        z.step(203)
        for k, (fa, fc) in enumerate(zip(fields(x), fields(z))):
            if x is a[2]:       # the general kernel's x chunk differs: rounding
                assert np.abs(fa - fc).max() <= 1e-5 * max(np.abs(f).max() for f in fields(z)[3 * (k // 3):3 * (k // 3) + 3])
            else:
                assert np.array_equal(fa, fc), k


@pytest.mark.parametrize("rows", ["2", "3"])
@pytest.mark.parametrize("flags", [0, G.BATCH_NO_TUNE])
def test_tiles_of_the_launches_per_variant_change_only_rounding(flags, rows, monkeypatch):
    steps = 160
    b = sims_for(CASES)
    with monkeypatch.context() as m:
        m.setenv("FDTD_ROWS", rows)
        a = sims_for(CASES)
    tb = G.Batch(b)                        # one launch
    with monkeypatch.context() as m:
        m.setenv("FDTD_ONE_LAUNCH", "0")
        ta = G.Batch(a, flags=flags)
    assert tb.tile(0)[2] <= 8 and (flags == 0 or ta.tile(0)[1] == int(rows))
    ta.run(steps)
    tb.run(steps)
    for i, (x, y) in enumerate(zip(a, b)):
        fx, fy = fields(x), fields(y)
        for g in (slice(0, 3), slice(3, 6)):
            scale = max(np.abs(f).max() for f in fy[g])
            for u, v in zip(fx[g], fy[g]):
                assert np.abs(u - v).max() <= 1e-5 * scale, (i, ta.tile(i))
