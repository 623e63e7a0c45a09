"""The runtime calls that the library's host code makes, on a stand-in for the
HIP runtime (fake_hip.cpp: host memory, kernels counted and not run).  Each test
runs its lines in a process of its own, where the stand-in is loaded first.

In those lines: D the package, hip the stand-in, calls(name) and launches(part)
its counts, lattice() a lattice with parameters and populations."""
import os
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

PREAMBLE = """
import ctypes, sys
import numpy as np
hip = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
for fn in ("calls", "launches", "live", "flags_up", "graph_nodes", "busy_used"):
    getattr(hip, "fake_hip_" + fn).restype = ctypes.c_int64
sys.path.insert(0, sys.argv[2])
import dlbc_amd as D

def calls(name):
    return hip.fake_hip_calls(name.encode())

def launches(part):
    return hip.fake_hip_launches(part.encode())

def live(device):
    return hip.fake_hip_live(device)

def fail(name, nth=1, code=1):
    hip.fake_hip_fail(name.encode(), nth, code)

def lattice(n, nc=2, sc=True, storage="f64", device=0):
    d, q = len(n), (19 if len(n) == 3 else 9)
    lat = D.Lattice(d, q, nc, n, storage=storage, device=device)
    lat.set_params([1.0] * nc, [[0.0 if i == j else 3.6 for j in range(nc)] for i in range(nc)],
                   None, None, None, "BDist2", "Exponential", sc)
    for f in range(nc):
        lat.init_fluid(f, "EqDist", [0.5], "BDist2")
    return lat
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake_hip") / "libfake_hip.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-fPIC", "-shared", "-pthread",
                    os.path.join(HERE, "fake_hip.cpp"), "-o", so], check=True)

    def go(lines):
        r = subprocess.run([sys.executable, "-c", PREAMBLE + textwrap.dedent(lines), so,
                            os.path.dirname(HERE)], capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, r.stdout + r.stderr
    return go


@pytest.mark.parametrize("n,nc,sc,steps", [((64, 64), 2, True, 33), ((64, 64), 1, False, 200),
                                           ((20, 20, 20), 2, True, 33), ((20, 20, 20), 1, False, 35),
                                           ((70, 80, 64), 2, True, 33)], ids=str)
def test_a_lattice_keeps_a_graph_of_each_buffer_parity(run, n, nc, sc, steps):
    run(f"""
    lat = lattice({n}, {nc}, {sc})
    for k in range(8):
        lat.step({steps}, graph=True)
    assert calls("hipGraphInstantiate") == 2, calls("hipGraphInstantiate")
    assert calls("hipGraphLaunch") == 8 * ({steps} // 32)
    lat.set_launch(512)  # new arguments: captured again
    lat.step(32, graph=True)
    assert calls("hipGraphInstantiate") == 3
    """)


@pytest.mark.parametrize("n,steps", [((120, 120, 120), 3), ((120, 120, 120), 4), ((16, 16, 16), 3)],
                         ids=str)
def test_a_batch_keeps_a_graph_of_each_flag_set(run, n, steps):
    run(f"""
    lats = [lattice({n}, storage="f32_shift") for _ in range(2)]
    batch = D.Batch(lats)
    batch.set_config(8, 64, 512, 2)
    for k in range(8):
        batch.step({steps}, graph=True)
    one = {n} == (120, 120, 120)  # one launch per step: flags in two sets
    assert launches("psi") == (0 if one else {steps} % 2 * 8 + 2), launches("psi")
    assert calls("hipGraphInstantiate") == (2 if one and {steps} % 2 else 1)
    assert calls("hipGraphLaunch") == 8 * ({steps} // 2)
    lats[0].set_params([1.0, 1.0], None, None, None, None, "BDist2", "Exponential", False)
    lats[1].set_params([1.0, 1.0], None, None, None, None, "BDist2", "Exponential", False)
    made = calls("hipGraphInstantiate")
    batch.step(2, graph=True)  # other kernels: captured again
    assert calls("hipGraphInstantiate") == made + 1
    """)


@pytest.mark.parametrize("storage,n,one", [
    ("f64", (100000, 10, 10), False), ("f64", (20000, 4, 4), False), ("f64", (4, 4, 65536), False),
    ("f64", (2500, 8, 16), True), ("f64", (25, 25, 520), True), ("f64", (41, 3, 2620), True),
    ("f64", (10, 11, 4096), False), ("f64", (15, 17, 4096), True), ("f64", (4, 4, 20000), False),
    ("f64", (8, 8, 16384), True), ("f64", (16, 8, 16385), False),
    ("f32_shift", (7000, 15, 16), False), ("f32_shift", (6100, 16, 16), True),
    ("f32_shift", (7, 9, 24569), False), ("f32_shift", (9, 10, 24569), True),
    ("f32_shift", (16, 16, 32768), True), ("f32_shift", (16, 16, 32769), False),
    ("f16_shift", (100000, 10, 10), False), ("f16_shift", (12000, 16, 16), False),
    ("f16_shift", (40000, 16, 16), True), ("f16_shift", (3200, 16, 32), True),
    ("f16_shift", (20, 20, 8192), False), ("f16_shift", (25, 26, 8192), True),
    ("f16_shift", (32, 32, 16384), True), ("f16_shift", (32, 32, 16385), False)], ids=str)
def test_thin_planes_and_long_rows_take_two_launches(run, storage, n, one):
    """A block of sites that meets more than two planes would wait for the whole
    lattice, and long rows for many blocks."""
    run(f"""
    lat = lattice({n}, storage="{storage}")
    lat.step(3)
    assert launches("split_psi") == {0 if one else 3}, launches("split_psi")
    assert launches("split_collide") == 3
    """)


@pytest.mark.parametrize("n,one", [((1000, 4, 4), True), ((4096, 4, 4), True), ((4097, 4, 4), False),
                                   ((4, 5, 32768), True), ((4, 5, 32769), False),
                                   ((7, 9, 24569), True)], ids=str)
def test_thin_planes_and_long_rows_of_a_batch_member(run, n, one):
    """A large member of such a shape decides for its batch, a small one does not."""
    run(f"""
    batch = D.Batch([lattice((128, 128, 96), storage="f32_shift"),
                     lattice({n}, storage="f32_shift")])
    batch.set_config(8, 64, 512, 2)
    batch.step(3, graph=False)
    assert launches("batch_split_collide") == 3
    assert launches("batch_split_psi") == {0 if one else 3}
    """)


@pytest.mark.parametrize("current", [0, 1])
def test_memory_is_made_on_the_device_of_its_lattice(run, current):
    """What is allocated after the creation of a lattice or a batch lies on its
    device, whichever the calling thread has current, and that one stays."""
    run(f"""
    lats = [lattice((70, 80, 64), device=k) for k in range(2)]
    shifted = [lattice((128, 128, 96), storage="f32_shift", device=k) for k in range(2)]
    tiled = [lattice((16, 16, 16), storage="f32_shift", device=k) for k in range(2)]
    batches = [D.Batch([lat]) for lat in shifted]
    for b in batches:
        b.set_config(8, 64, 512, 2)
    hip.hipSetDevice({current})
    now = ctypes.c_int(-1)

    def lies_on(device, work, count):
        before = live(device), live(1 - device)
        work()
        assert (live(device) - before[0], live(1 - device) - before[1]) == (count, 0), (
            device, live(device) - before[0], live(1 - device) - before[1])
        hip.hipGetDevice(ctypes.byref(now))
        assert now.value == {current}

    for k in (0, 1):
        lies_on(k, lambda: lats[k].step(1), 2)  # order and flags
        lies_on(k, lambda: batches[k].step(1), 3)  # and the batch's items
        lies_on(k, lambda: lats[k].step(1), 0)
        tiled[k].set_schedule("fused")
        lies_on(k, lambda: tiled[k].step(1), 1)  # its items
        lies_on(k, lambda: tiled[k].density(0), 2)  # a slot: its memory and event
        before = live(1 - k)
        lats[k].density(0)  # scratch, and slots as the threads take them
        assert live(1 - k) == before
    del lats, shifted, tiled, batches, b
    import gc
    gc.collect()
    assert live(0) == 0 and live(1) == 0
    """)


FAILURES = [("hipLaunchKernel", 1), ("hipLaunchKernel", 2), ("hipStreamEndCapture", 1),
            ("hipGraphInstantiate", 1), ("hipGraphLaunch", 1), ("hipGraphLaunch", 2),
            ("hipGetLastError", 1), ("hipGetLastError", 2)]


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("what", ["lattice", "batch"])
def test_flags_are_down_after_a_call_that_failed(run, what, graph):
    """Every launch of the one-launch step starts with its flags down, also after
    a call that failed before, within or after a capture, and no graph that is
    short of a launch is kept."""
    run(f"""
    for name, nth in {FAILURES}:
        for before in (0, 1, 32, 33):
            if "{what}" == "lattice":
                it = lattice((70, 80, 64))
            else:
                it = D.Batch([lattice((128, 128, 96), storage="f32_shift")])
                it.set_config(8, 64, 512, 2)
                if before == 33:
                    it.autotune()
                    it.set_config(8, 64, 512, 2)
            it.step(before, graph={graph})
            it.synchronize()
            fail(name, nth)
            try:
                it.step(65, graph={graph})
            except D.DlbcError:
                pass
            fail(name, 1 << 30)  # not planned any longer
            for k in (1, 64, 33, 2, 65):
                it.step(k, graph={graph})
                if {graph} and k > 1:
                    assert hip.fake_hip_graph_nodes() == (32 if "{what}" == "lattice" else 2)
            assert hip.fake_hip_flags_up() == 0, (name, nth, before)
    """)


@pytest.mark.parametrize("n,nc,sc,steps,per", [((64, 64), 1, False, 35, 8), ((200, 200), 1, False, 6, 4),
                                               ((64, 64), 1, False, 3, 8), ((64, 64), 1, False, 16, 8),
                                               ((64, 64), 2, True, 5, 1), ((600, 600), 1, False, 5, 1),
                                               ((20, 20, 20), 2, True, 3, 1)], ids=str)
def test_timed_steps_launch_what_steps_launch(run, n, nc, sc, steps, per):
    run(f"""
    lat = lattice({n}, {nc}, {sc})
    counts = []
    for work in (lat.step, lat.step_timed):
        before = [launches(k) for k in ("", "k_single_multi")]
        out = work({steps})
        counts.append([launches(k) - b for k, b in zip(("", "k_single_multi"), before)])
    assert counts[0] == counts[1], counts
    assert counts[0][1] == ({steps} // {per} if {per} > 1 else 0)
    kernels = out[1]
    if {per} > 1:  # a launch takes 1 ms on the stand-in
        want = {{"stream_collide": 1.0 if {steps} % {per} else 0.0}}
        if {steps} >= {per}:
            want["stream_collide_steps"] = 1.0
        assert kernels == want, kernels
    else:
        assert set(kernels.values()) == {{1.0}} and "" not in kernels
    """)


@pytest.mark.parametrize("storage,n", [("f64", (70, 80, 64)), ("f32_shift", (128, 128, 96))])
def test_timed_steps_start_with_the_tables_made(run, storage, n):
    run(f"""
    lat = lattice({n}, storage="{storage}")
    before = live(0)
    fail("hipEventRecord", 1)  # the one that starts the time
    try:
        lat.step_timed(1)
        assert False
    except D.DlbcError:
        pass
    assert live(0) == before + 2
    """)


@pytest.mark.parametrize("storage", ["f32_shift", "f16_shift"])
def test_the_large_batch_takes_one_launch_per_step(run, storage):
    from test_split_one_launch import BATCH
    run(f"""
    batch = D.Batch([lattice(n, storage="{storage}") for n in {BATCH}])
    batch.set_config(8, 64, 512, 2)
    batch.step(5, graph=False)
    assert launches("batch_split_collide") == 5 and launches("batch_split_psi") == 0
    batch = D.Batch(batch.members[:3])  # 5,907 blocks
    batch.set_config(8, 64, 512, 2)
    batch.step(5, graph=False)
    assert launches("batch_split_collide") == 10 and launches("batch_split_psi") == 5
    """)


@pytest.mark.parametrize("n", [(16, 16, 16), (40, 40, 40)], ids=str)
@pytest.mark.parametrize("name", ["hipMemcpyAsync", "hipEventRecord", "hipEventSynchronize"])
@pytest.mark.parametrize("stuck", [False, True])
def test_pinned_memory_is_not_used_again_while_a_copy_may_be_under_way(run, n, name, stuck):
    """After a transfer that failed between its copy and the wait for it, also
    where the stream cannot be waited for."""
    run(f"""
    pop = np.random.default_rng(1).random({n} + (19,))
    for nth in (1, 2, 3):
        a, b = lattice({n}), lattice({n})
        for work in (lambda: a.upload_population(0, pop), lambda: a.population(0)):
            fail("{name}", nth)
            if {stuck}:
                fail("hipStreamSynchronize", 0)
            try:
                work()
            except D.DlbcError:
                pass
            fail("{name}", 1 << 30)
            fail("hipStreamSynchronize", 1 << 30)
            b.upload_population(0, pop)
            b.population(0)
        del a, b
    assert hip.fake_hip_busy_used() == 0, hip.fake_hip_busy_used()
    """)


@pytest.mark.parametrize("n,nc,tile", [
    ((64, 64), 2, True), ((400, 400), 2, True), ((2048, 2048), 2, False), ((3001, 3001), 1, False),
    ((1024, 1024), 3, True), ((1225, 1225), 3, False), ((1225, 1225), 4, True),
    ((50000, 2), 2, False), ((24000, 4), 3, False), ((3, 500000), 4, False), ((4096, 2), 2, True),
    ((2, 8192), 1, True), ((24000, 16), 4, True), ((24000, 13), 4, True), ((24000, 12), 4, False)],
    ids=str)
def test_tiles_of_a_d2q9_step_are_mostly_sites(run, n, nc, tile):
    """Thin lattices, of whose tiles most cells are no sites, and large ones take
    two launches per step."""
    run(f"""
    lat = lattice({n}, {nc})
    lat.step(3)
    assert launches("k_tile_step") == {3 if tile else 0}
    assert launches("5k_psi") == {0 if tile else 3}
    """)


@pytest.mark.parametrize("n,per", [((64, 64), 8), ((2000, 2), 8), ((256, 256), 4), ((2000, 17), 4),
                                   ((400, 400), 4), ((4000, 20), 4), ((4706, 17), 1),
                                   ((17, 4706), 1), ((500, 500), 1)], ids=str)
def test_steps_of_a_launch(run, n, per):
    """More than one round of workgroups only where their tiles are mostly sites."""
    run(f"""
    lat = lattice({n}, 1, False)
    lat.step(8)
    assert launches("k_single") == 8 // {per}, launches("k_single")
    """)


@pytest.mark.parametrize("n,nt", [((96, 96, 96), 0), ((99, 99, 99), 0), ((100, 100, 100), 1),
                                  ((1400, 1400), 0), ((1500, 1500), 1)], ids=str)
@pytest.mark.parametrize("solid", [0, 1])
def test_single_component_stores_past_the_cache(run, n, nt, solid):
    """Nontemporal stores (the kernel's last template argument) from where both
    buffers no longer stay in the memory-side cache."""
    run(f"""
    lat = lattice({n}, 1, False)
    if {solid}:
        mask = np.zeros({n}, np.int32)
        mask[0] = 1
        lat.upload_mask(mask)
    lat.step(2)
    assert launches("k_singleI") == launches("Lb{solid}ELb{nt}EEEvPK") == 2
    """)
