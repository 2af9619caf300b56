"""Point-monitor records, taken by the next step's line launch within a call and
by a launch of their own after a call's last step: the same values whatever
the calls' lengths, and those of the fields read back; on the one-launch step,
on streams, on the general kernel; capacity reached in the middle of a call;
with an adjoint's own records running beside them."""
import numpy as np
import pytest

import fdtd_amd
from conftest import small_params

pytestmark = pytest.mark.gpu


def spectrum(s):
    return s.point_spectrum([3e14, 5e14, 7e14])[1]


@pytest.mark.parametrize("env", [{}, {"FDTD_ONE_LAUNCH": "0"}, {"FDTD_PATH": "general"}])
@pytest.mark.parametrize("cap", [200, 33])
def test_records_do_not_depend_on_the_calls(env, cap, monkeypatch):
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    p = small_params(fdtd_amd)
    out = []
    for calls in ([60], [1] * 60, [7, 1, 25, 2, 25]):
        s = fdtd_amd.Simulation(p)
        rng = np.random.default_rng(0)
        for c in range(3):
            s.set_field(c, (rng.standard_normal(s.shape) * 0.1).astype(np.float32))
        at = [e // 2 + 1 for e in s.shape]
        s.set_point_monitor(at, cap)
        seen = []
        for n in calls:
            s.step(n)
            seen.append([s.get_field(c)[tuple(at)] for c in range(3)] if len(calls) == 60 else None)
        out.append(spectrum(s))
        if len(calls) == 60:
            t = np.arange(1, min(cap, 60) + 1)
            w = np.exp(2j * np.pi * np.outer([3e14, 5e14, 7e14], t) * s.info.dt)
            want = w @ np.array(seen, float)[:min(cap, 60)]
            assert np.abs(out[-1] - want).max() <= 1e-12 * np.abs(want).max()
    assert np.abs(out[0]).max() > 0
    assert np.array_equal(out[0], out[1]) and np.array_equal(out[0], out[2])


@pytest.mark.parametrize("ckpt", [0, 20])
def test_monitor_beside_the_adjoint(ckpt):
    p = small_params(fdtd_amd, ncpml=5, n=20, sphere=0)
    rho = np.random.default_rng(1).uniform(0.1, 0.9, (4, 4, 3)).astype(np.float32)
    out = []
    for adj in (True, False):
        s = fdtd_amd.Simulation(p)
        c = [e // 2 for e in s.shape]
        s.set_design([v - 2 for v in c], rho)
        rng = np.random.default_rng(0)
        for q in range(3):
            s.set_field(q, (rng.standard_normal(s.shape) * 0.1).astype(np.float32))
        s.set_point_monitor(c, 100)
        if adj:
            s.adjoint(50, (c[0], c[1], c[2] + 4), [4e14], checkpoint=ckpt)
        else:
            s.step(50)
        s.step(10)
        out.append(spectrum(s))
    assert np.array_equal(out[0], out[1])
