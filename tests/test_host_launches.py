"""The host code alone, on a machine without a GPU: the library runs in a child
process over a stand-in for the HIP runtime (hip_stub.cpp), and the tests look
at the kernels that a call launches and at the handle's own state."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
PACKAGE = os.path.join(os.path.dirname(HERE), "fdtd-cuda_amd")


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("stub") / "hip_stub.so")
    subprocess.run(["g++", "-shared", "-fPIC", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-o", so,
                    os.path.join(HERE, "hip_stub.cpp")], check=True)
    return so


def run(stub, tmp_path, code, env=()):
    """Launches of the code after its last mark() as (kernel, grid, block), and what it printed."""
    log = tmp_path / "launches"
    log.write_text("")
    head = (f"import sys, ctypes; sys.path[:0] = [{PACKAGE!r}, {HERE!r}]\n"
            "import fdtd_amd as G\nfrom conftest import small_params\n"
            f"stub = ctypes.CDLL({stub!r})\nmark = lambda: open({str(log)!r}, 'w').close()\n"
            f"launched = lambda kernel: open({str(log)!r}).read().count(kernel)\n")
    kept = {k: v for k, v in os.environ.items() if not k.startswith("FDTD_")}
    r = subprocess.run([sys.executable, "-c", head + code], capture_output=True, text=True, timeout=300,
                       env={**kept, "LD_PRELOAD": stub, "HIP_STUB_LOG": str(log), **dict(env)})
    assert r.returncode == 0, r.stderr
    launches = [line.split("\t") for line in log.read_text().splitlines()]
    return [(k, *(tuple(int(x) for x in v.split()) for v in (g, b))) for k, g, b in launches], r.stdout


PERIODIC = """
p = small_params(G, sphere=0)
p.periodic_xy, p.NcpmlX, p.NcpmlY, p.NcpmlZ = 1, 0, 0, 8
p.NCELLX, p.NCELLY, p.NCELLZ = 6, 5, 80
p.tfsf_inset, p.sca_offset, p.dft_stride = 10, {offset}, 1
s = G.Simulation(p)
k0 = s.info.tfsf[2] + {at}
s.add_layer(k0, k0 + {thick})
mark()
s.step(1)
"""


@pytest.mark.parametrize("offset,at,thick,apart", [(5, 1, 4, True), (-3, 1, 5, False), (-3, 3, 1, False), (-3, 2, 1, False),
                                                   (-3, 4, 2, False), (-3, 5, 4, True), (-8, 1, 4, True)])
def test_periodic_sample_follows_a_layer_on_its_plane(stub, tmp_path, offset, at, thick, apart):
    """The reflection plane is tfsf - offset: on or beside the layer's box, the
    sample is a launch after the box's; apart from it, they share one."""
    launches, _ = run(stub, tmp_path, PERIODIC.format(offset=offset, at=at, thick=thick))
    names = [k for k, _, _ in launches]
    tail = ["k_post"] if apart else ["k_post", "k_dft_sample_split"]
    assert names == ["k_per_h", "k_per_e"] + tail
    cells = 6 * 5
    blocks = -(-cells * (thick + 2) // 256) + (-(-4 * cells // 256) if apart else 0)
    assert launches[2][1] == (blocks, 1, 1)


@pytest.mark.parametrize("env", [{}, {"FDTD_ONE_LAUNCH": "0"}, {"FDTD_PATH": "general"}])
def test_a_failed_step_leaves_no_record_behind(stub, tmp_path, env):
    """Whichever launch of three steps fails, the handle holds no pointer into
    the point monitor's buffer afterwards, and the records of the steps before
    are taken."""
    launches, out = run(stub, tmp_path, """
for n in range(1, 40):
    s = G.Simulation(small_params(G))
    s.set_point_monitor((5, 6, 7), 10)
    mark()
    stub.stub_fail_launch(n)
    try:
        s.step(3)
    except G.FDTDError as e:
        assert 'stub error' in str(e)
        print(n, stub.stub_pending_records(s.h), launched('k_probe'))
    else:
        break
    s.close()
""", env)
    rows = [tuple(map(int, line.split())) for line in out.splitlines()]
    assert len(rows) >= 7
    assert all(pending == 0 for _, pending, _ in rows), rows
    assert rows[0][2] == 0 and rows[-2][2] == 1, rows   # the last launch of all is the record's own


@pytest.mark.parametrize("nz,kernel,waves", [(24, "k_step_batch<12>", 4), (200, "k_step_batch<12>", 12), (270, "k_step_batch<16>", 15),
                                             (330, "k_step_batch<12>", 12), (400, "k_step_batch<16>", 8),
                                             (600, "k_step_batch<12>", 12), (800, "k_step_batch<16>", 16)])
def test_batch_blocks_fill_a_compute_unit(stub, tmp_path, nz, kernel, waves):
    """Blocks of the batched one-launch step by column height: 5 waves a column
    in blocks of 15, 2 (alone in their batch) in blocks of 4, and the instance by
    the waves that fit a compute unit."""
    launches, _ = run(stub, tmp_path, f"""
p = small_params(G, sphere=0)
p.NCELLZ = {nz}
s = [G.Simulation(p) for _ in range(2)]
b = G.Batch(s, flags=G.BATCH_NO_GRAPH)
mark()
b.run(1)
""")
    assert launches[0][0] == kernel and launches[0][2] == (64, waves, 1), launches


@pytest.mark.parametrize("n,one", [((350, 364), True), ((354, 364), False)])
def test_batch_leaves_one_launch_where_fdtd_step_does(stub, tmp_path, n, one):
    """One launch for a batch only up to the 50 M cells a simulation that fdtd_step's rule has."""
    launches, out = run(stub, tmp_path, f"""
sims = []
for nx, nz in ((24, 24), {n}):
    p = small_params(G, sphere=0, nfreq=1)
    p.NCELLX = p.NCELLY = nx
    p.NCELLZ = nz
    sims.append(G.Simulation(p))
print(sims[1].info.NX * sims[1].info.NY * sims[1].info.NZ, sims[1].get_info().tile[6])
b = G.Batch(sims, flags=G.BATCH_NO_GRAPH | G.BATCH_NO_TUNE)
mark()
b.run(1)
""")
    cells, streams = map(int, out.split())
    assert (cells <= 50_000_000) == one and (streams == 0) == one
    assert any(k.startswith("k_step_batch") for k, _, _ in launches) == one, launches
    assert any(k.startswith("k_rows_batch") for k, _, _ in launches) != one


@pytest.mark.parametrize("path", ["general", "rows"])
@pytest.mark.parametrize("fuse,own", [(None, 1), ("1", 1), ("0", 9)])
def test_injection_has_its_own_launch_where_the_switch_says(stub, tmp_path, path, fuse, own):
    """FDTD_ADJ_FUSE_INJECT=0 gives every injection of a reverse sweep a launch
    of its own on either transposed kernel; else only the first one has."""
    env = {"FDTD_ADJ_PATH": "general"} if path == "general" else {}
    if fuse:
        env["FDTD_ADJ_FUSE_INJECT"] = fuse
    launches, _ = run(stub, tmp_path, """
import numpy as np
s = G.Simulation(small_params(G, n=22, ncpml=5, sphere=0))
s.set_design((14, 15, 16), np.full((4, 3, 2), 0.5, np.float32))
mark()
s.adjoint(9, (17, 17, 14), [4e14], checkpoint=4)
""", env)
    names = [k for k, _, _ in launches]
    assert names.count("k_adj_inject") == own
    assert any(k.startswith("k_adj_step") for k in names) == (path == "general")


@pytest.mark.parametrize("nz", [24, 200, 270, 331, 420, 600])
@pytest.mark.parametrize("env,one", [({}, True), ({"FDTD_TILES": "1"}, True), ({"FDTD_CONCURRENT": "0"}, False),
                                     ({"FDTD_ONE_LAUNCH": "0"}, False)])
def test_info_names_the_launch_that_runs(stub, tmp_path, nz, env, one):
    """fdtd_grid_info.tile: the row tiles of the launch, and tile[5] 0 exactly
    where every piece is in one launch (tile[6] is 0 on one stream as well)."""
    launches, out = run(stub, tmp_path, f"""
p = small_params(G, sphere=0)
p.NCELLZ = {nz}
s = G.Simulation(p)
print(*s.get_info().tile, s.info.NZ)
mark()
s.step(1)
""", env)
    *tile, nz = map(int, out.split())
    assert (tile[5] == 0) == one and (tile[6] == 0) == (one or "FDTD_CONCURRENT" in env)
    columns = next(w for w in (2, 3, 4, 5, 6, 8, 12, 16) if 64 * w - 2 >= nz + 1)
    kernel = "k_step_all" if one else "k_step_rows"
    blocks = [b[1] for k, _, b in launches if k.startswith(kernel)]
    assert columns * tile[3] in blocks and columns * tile[4] in blocks, (tile, launches)
    if one:
        assert len(blocks) == 1


@pytest.mark.parametrize("env", [{}, {"FDTD_ONE_LAUNCH": "1"}])
def test_more_than_4_gb_of_psi_keep_the_row_blocked_kernel(stub, tmp_path, env):
    """31 CPML layers of a flat grid: each array within 4 GB, all together not."""
    launches, out = run(stub, tmp_path, """
p = small_params(G, sphere=0, nfreq=1, ncpml=31)
p.NCELLX = p.NCELLY = 1577
s = G.Simulation(p)
print(s.info.NX, s.info.NZ, s.info.fused_path, s.get_info().tile[5])
mark()
s.step(1)
""", env)
    n, nz, path, corners = map(int, out.split())
    assert 4 * (n + 2) * (n + 2) * (nz + 11) < 1 << 32
    assert 4 * (4 * 62 + 2 * 64) * (n * n + 2 * n * nz) > 1 << 32
    assert path == 1 and corners > 0
    assert any(k.startswith("k_step_rows") for k, _, _ in launches)


@pytest.mark.parametrize("read", ["s.get_field(2)", "s.checkpoint()"])
def test_a_read_out_behind_queued_steps_does_not_keep_the_cores_busy(stub, tmp_path, read):
    """The threads that move a field to the caller poll for its bytes, so they
    start once the work queued before has ended (0.4 s of it here)."""
    _, out = run(stub, tmp_path, f"""
import time
s = G.Simulation(small_params(G, n=120, nfreq=1, sphere=0))
{read}
s.step(1)
idle = time.process_time()
{read}
idle = time.process_time() - idle
stub.stub_queue(400)
queued = time.process_time()
{read}
print(idle, time.process_time() - queued)
""")
    idle, queued = map(float, out.split())
    assert queued - idle < 0.2, (idle, queued)


@pytest.mark.parametrize("shape", [(24, 24, 24), (300, 22, 24), (22, 300, 24), (24, 22, 300), (140, 150, 20)])
def test_tfsf_launches_hold_the_rows_of_the_planes(stub, tmp_path, shape):
    """Four planes of t0 - 1 .. t1 + 1 per axis after the update (three of t0 - 1 ..
    t1 between separate calls), in rows of 64 cells along the faster axis and
    four rows a block, each axis by its own extents."""
    launches, out = run(stub, tmp_path, f"""
p = small_params(G, sphere=0)
p.NCELLX, p.NCELLY, p.NCELLZ = {shape}
s = G.Simulation(p)
print(s.info.NX, s.info.NY, s.info.NZ, *s.info.tfsf)
mark()
s.step(2)
s.tfsf()
""")
    size, t0 = [int(x) for x in out.split()[:3]], [int(x) for x in out.split()[3:6]]
    t1 = [n - t for n, t in zip(size, t0)]

    def blocks(planes, past):
        n = [b - a + 2 + past for a, b in zip(t0, t1)]
        rows = sum(planes * n[0 if a else 1] * -(-n[1 if a == 2 else 2] // 64) for a in range(3))
        return -(-rows // 4)
    posts = [g for k, g, _ in launches if k == "k_post"]
    assert posts[1] == (blocks(4, 1), 1, 1)      # the second step takes no sample
    assert [g for k, g, _ in launches if k == "k_tfsf_split"] == [(blocks(3, 0), 1, 1)]


def test_small_read_outs_wait_once(stub, tmp_path):
    """Blocks below the size that threads move: one wait for a field, one for a
    whole checkpoint of small arrays, not one each."""
    _, out = run(stub, tmp_path, """
s = G.Simulation(small_params(G, nfreq=1, sphere=0))
s.set_point_monitor((5, 6, 7), 10)
for f in (lambda: s.get_field(0), lambda: s.checkpoint()):
    n = stub.stub_waits()
    f()
    print(stub.stub_waits() - n)
""")
    assert [int(x) for x in out.split()] == [1, 1]


@pytest.mark.parametrize("nz,device", [(40, False), (133, False), (134, True), (682, True), (683, False)])
def test_incident_line_is_replayed_where_that_is_faster(stub, tmp_path, nz, device):
    """Lines of 6 NCELLZ cells: on the device from 800 to 4096."""
    launches, _ = run(stub, tmp_path, f"""
p = small_params(G, sphere=0, nfreq=2)
p.periodic_xy, p.NcpmlX, p.NcpmlY, p.NcpmlZ = 1, 0, 0, 8
p.NCELLX, p.NCELLY, p.NCELLZ, p.tfsf_inset = 8, 8, {nz}, 10
s = G.Simulation(p)
s.step(20)
mark()
s.reflectance()
""")
    assert any(k.startswith("k_line_replay") for k, _, _ in launches) == device


@pytest.mark.parametrize("sizes,waves", [([(1, 24), (1, 150)], [12]), ([(1, 24), (1, 300)], [12, 15]), ([(48, 24), (1, 150)], [4, 12]),
                                         ([(48, 24), (34, 150)], [12]), ([(3, 24)], [4]), ([(2, 24), (2, 101)], [4])])
def test_batch_of_short_columns_takes_small_blocks(stub, tmp_path, sizes, waves):
    """Columns of 2 waves in blocks of 4 where they are the whole batch, or most of
    one that fills the device; else in the blocks of 12 of the other heights."""
    launches, _ = run(stub, tmp_path, f"""
s = []
for n, nz in {sizes}:
    for _ in range(n):
        p = small_params(G, sphere=0, nfreq=1)
        p.NCELLZ = nz
        s.append(G.Simulation(p))
b = G.Batch(s, flags=G.BATCH_NO_GRAPH)
mark()
b.run(1)
""")
    assert sorted(b[1] for k, _, b in launches if k.startswith("k_step_batch")) == waves, launches
