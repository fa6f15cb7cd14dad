"""The host code between the C API and the device, run without a GPU: a HIP
runtime in host memory (fake_hip.c) stands in for the real one, so that what
the library allocates, launches and times can be counted.  Each test is a
program of its own, since the stand-in has to be loaded ahead of the library.
"""
import os
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
ROCM = "/opt/rocm/include"

pytestmark = pytest.mark.skipif(not os.path.isdir(os.path.join(ROCM, "hip")), reason="no HIP headers")

PRELUDE = """
import ctypes as C, sys
fake = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
import numpy as np
import albba_amd as A

def get(name, ctype=C.c_longlong, n=0):
    return (ctype * n).in_dll(fake, name) if n else ctype.in_dll(fake, name)

def kernels():
    return C.string_at(C.addressof(get("fake_log", C.c_char, 1 << 22))).decode().split()

def empty(n):
    # no entries: the stand-in runs no kernel, so a built layout holds none
    return A.Graph.from_arrays(np.zeros(n + 1, np.int64), np.zeros(0, np.int32), symmetric=True)

def levels(frontier, edges):
    get("fake_levels", C.c_int).value = len(frontier)
    get("fake_frontier", n=65)[:len(frontier)] = frontier
    get("fake_edges", n=65)[:len(edges)] = edges

live = lambda d=0: get("fake_live_bytes", n=2)[d]
blocks = lambda d=0: get("fake_live_blocks", n=2)[d]
"""


@pytest.fixture(scope="session")
def fake_hip(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake_hip") / "fake_hip.so")
    subprocess.run(["gcc", "-O1", "-fPIC", "-shared", "-std=gnu11", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__=1",
                    "-I" + ROCM, "-I" + os.path.join(ROOT, "include"), "-o", so, os.path.join(HERE, "fake_hip.c")],
                   check=True)
    return so


@pytest.fixture
def program(fake_hip):
    def run(body):
        r = subprocess.run([sys.executable, "-c", PRELUDE + textwrap.dedent(body), fake_hip], cwd=ROOT,
                           capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, r.stdout + r.stderr

    return run


def test_kept_blocks_are_few(program):
    """Freed device blocks that a context keeps are bounded in number and
    bytes: closing thousands of small graphs gives most of them back."""
    program("""
        ctx = A.Context(0)
        gs = [A.DeviceGraph.build(ctx, empty(100), 64, 64, 1) for _ in range(600)]
        for g in gs:
            g.close()
        assert blocks() <= 4096, blocks()
        # and they are used again: a graph like the last one takes none from
        # the device
        A.DeviceGraph.build(ctx, empty(100), 64, 64, 1).close()
        before = blocks()
        g = A.DeviceGraph.build(ctx, empty(100), 64, 64, 1)
        assert blocks() == before
        g.close()
        ctx.close()
        assert blocks() == 0 and live() == 0
    """)


def test_kept_blocks_go_to_other_contexts(program):
    """A context that runs out of device memory gets the blocks that the
    device's other contexts keep; trim gives a context's own back."""
    program("""
        get("fake_capacity").value = 1 << 30
        a, b = A.Context(0), A.Context(0)
        other = A.Context(1)
        other.bench_copy(300 << 20, 1)
        a.bench_copy(400 << 20, 1)
        assert live() >= 800 << 20
        b.bench_copy(300 << 20, 1)
        assert live(1) >= 600 << 20  # another device's are left alone
        a.bench_copy(400 << 20, 1)
        # what does not fit an empty device fails as before
        try:
            b.bench_copy(600 << 20, 1)
            raise SystemExit("1.2 GB on a device of 1 GB")
        except A.AlbbaError as e:
            assert e.code == -7
        b.trim()
        assert live() == 0
        a.bench_copy(200 << 20, 1)
        assert live() == 400 << 20
        a.trim()
        assert live() == 0
        a.close()
        assert A.lib().albba_ctx_trim(None) == -1
        b.bench_copy(500 << 20, 1)
        b.close()
        assert live() == 0
    """)


def test_allocating_makes_the_device_current(program):
    """Two devices in one thread: a call that allocates makes its context's
    device the current one, also where the memory is a kept block."""
    program("""
        a, b = A.Context(0), A.Context(1)
        for _ in range(3):
            a.bench_copy(1 << 20, 1)
            b.bench_copy(1 << 20, 1)
        assert get("fake_wrong_device", C.c_int).value == 0
    """)


@pytest.mark.parametrize("count", [5, 200, 5000])
def test_batch_memory_of_small_graphs(program, count):
    """A batch of small graphs takes the memory of its graphs: per instance
    four bitmaps, the found list, keys, results and a control block; what the
    teams' unfilled reservations (16 KB a workgroup) and barrier slots (3 KB) add is
    bounded by the workgroups of one launch, whatever the number of graphs."""
    program(f"""
        count = {count}
        ctx = A.Context(0)
        g = A.DeviceGraph.build(ctx, empty(1000), 64, 64, 1)
        ctx.trim()
        before = live()
        b = A.Batch(ctx, [g] * count)
        n, npos = 1000, 1024
        own = 4 * 8 * (npos // 64) + (4 + 8) * npos + 8 * n + 8 * 32
        workgroups = 512  # the stand-in's 256 compute units hold two each
        slack = workgroups * (2 * 2048 * 4 + 6 * 64 * 8)
        assert live() - before <= count * own + slack, (live() - before, count * own, slack)
        b.close()
        ctx.close()
    """)


# a BFS that pushes on every level: a frontier beyond the one-block scan, one
# with too many edges for its queue to be listed, and the push after that
PUSHES = "levels([1, 10, 9000, 11000, 11500, 50], [5, 9000, 30000, 11000, 11900, 100])"


def test_best_times_a_push_as_it_is_deployed(program):
    """The BEST policy's time of a push covers the kernels that the same push
    costs in the level loop (every kernel takes 1 ms here): no scan of a queue
    that was listed with its prefix, and no queue listed where the loop lists
    none."""
    program(f"""
        g = A.DeviceGraph.build(A.Context(0), empty(300000), 64, 4096, 1)
        {PUSHES}
        done = get("fake_finalizes", C.c_int)
        loop = g.bfs(0, policy=A.SWITCH_HEURISTIC, time_levels=True, small_frontier_edges=0, results=False)
        caps = list(get("fake_build_max", n=4096)[:done.value])
        done.value = 0
        best = g.bfs(0, policy=A.SWITCH_BEST, timing_reps=1, results=False)
        assert list(loop["choice"]) == [A.CHOICE_PUSH] * 6 == list(best["choice"])
        assert list(best["choice_ms"][:, A.CHOICE_PUSH]) == list(loop["level_ms"]), (best["choice_ms"], loop["level_ms"])
        # the trial of each level, with the loop's limit, then the committed
        # push, which lists every queue
        assert list(get("fake_build_max", n=4096)[:done.value]) == [x for c in caps for x in (c, 2**63 - 1)]
    """)


def test_fixed_pushes_scan_no_queue(program):
    """A queue that the last push listed has its degree prefix: the pushes of
    the FIXED policy do not scan it again."""
    program(f"""
        g = A.DeviceGraph.build(A.Context(0), empty(300000), 64, 4096, 1)
        {PUSHES}
        fake.fake_log_reset()
        r = g.bfs(0, policy=A.SWITCH_FIXED, fixed_choice=A.CHOICE_PUSH, results=False)
        assert r["num_levels"] == 6
        assert not [k for k in kernels() if "k_scan" in k]
        # a pull in front of a push: the queue and its prefix come from the bitmap
        fake.fake_log_reset()
        g.bfs(0, policy=A.SWITCH_SCRIPT, script=[0, 1, 0, 0, 2, 0], results=False)
        assert not [k for k in kernels() if "k_scan" in k]
    """)


def test_conv_time_is_the_layout_build(program):
    """conv_time of the reference's entry point is the SELL build: what the
    device build reports for the same matrix (kernels take 1 ms here), without
    the upload and the BFS state around it."""
    program("""
        g = empty(1000)
        sigma = 16384  # the reference's sigma_window
        want = A.DeviceGraph.build(A.Context(0), g, 64, sigma, 1).build_report["build_ms"]
        assert want >= 5 and want == int(want)
        levels([1], [0])
        r = A.run_custom_bfs_test(1000, np.zeros(1001, np.int32), np.zeros(0, np.int32))
        assert r["conv_time"] == want, (r["conv_time"], want)
    """)


def test_upload_time_is_the_copy(program):
    """upload_ms of a build is the CSR's way to the device, without the
    allocation of its arrays (here 50 ms each)."""
    program("""
        get("fake_malloc_us", C.c_int).value = 50000
        t = A.DeviceGraph.build(A.Context(0), empty(10), 64, 64, 1).build_report["upload_ms"]
        assert t < 50, t
    """)


def test_without_pinned_memory(program):
    """Where the pinned level log and the copies' stages cannot be allocated, a
    small graph's BFS runs in the level loop and results come by plain copies;
    where they can again, in one workgroup."""
    program("""
        ctx = A.Context(0)
        get("fake_pinned_max").value = 1 << 18
        g = A.DeviceGraph.build(ctx, empty(5000), 64, 64, 1)
        big = A.DeviceGraph.build(ctx, empty(1 << 20), 64, 64, 1)
        levels([1, 3], [2, 0])
        fake.fake_log_reset()
        r = g.bfs(0)
        assert r["num_levels"] == 2 and r["level"].size == 5000
        assert [k for k in kernels() if "k_bfs_reset" in k] and not [k for k in kernels() if "k_bfs_one" in k]
        assert big.bfs(0)["parent"].size == 1 << 20
        get("fake_pinned_max").value = 1 << 40
        fake.fake_log_reset()
        g.bfs(0)
        assert [k for k in kernels() if "k_bfs_one" in k] and not [k for k in kernels() if "k_bfs_reset" in k]
    """)
