"""What the library's host code asks of the HIP runtime, on the CPU: the runtime's calls are those of hip_host.cpp,
which keeps every stream's work waiting until something synchronises with it and runs no kernels."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

# the runtime before the library, in a process of its own, without torch
PRELUDE = """
import ctypes, resource, sys, time
H = ctypes.CDLL({runtime!r}, ctypes.RTLD_GLOBAL)
sys.path[:0] = [{root!r}, {here!r}]
import numpy as np
import gpu_phs_amd as G
from gpu_phs_amd import workloads as W
H.hip_host_elapsed.argtypes = [ctypes.c_double, ctypes.c_double]
H.hip_host_groups.restype = H.hip_host_most_lds.restype = ctypes.c_int64

def i(v):
    return ctypes.byref(ctypes.c_int(v))

def p(a):
    return a.ctypes.data_as(ctypes.c_void_p)

def launches():
    text = ctypes.create_string_buffer(1 << 20)
    H.hip_host_launches(text, len(text))
    return text.value.decode().split()

class Array:
    # a segment's array: host memory, as the runtime's device memory is
    def __init__(self, shape, dtype=np.float64):
        self.a = np.zeros(shape, dtype)
        self.shape, self.dtype = self.a.shape, self.a.dtype
    def is_contiguous(self):
        return True
    def data_ptr(self):
        return self.a.ctypes.data

class Stream:
    cuda_stream = 0

def plan(proc, counts, **config):
    ph, segs = G.ProcessHandle(proc), []
    for c, n in enumerate(counts):
        if n:
            segs.append((ph, c, G.EventBuffers(Array((n, proc.n_x)), Array((n, proc.n_out, 4)), Array(n), Array(n),
                                               Array(n, np.uint8))))
    return G.Plan(segs, **config)

def whizard(proc, counts):
    # the host program's calls up to the first event, and the call that generates
    L, nc, n = G.lib(), proc.n_channels, sum(counts)
    L.c_whizard_set_particle_structure(i(nc), i(nc), i(1), i(proc.n_x), i(proc.n_in), i(proc.n_out))
    flv = np.ascontiguousarray(proc.flv_masses)
    L.c_whizard_set_flavors(p(flv), p(np.zeros_like(flv)))
    L.c_whizard_init_mappings()
    L.c_whizard_init_tree_structures()
    for c in range(nc):
        ids, m, w, d1, d2, hc = (np.ascontiguousarray(a[c]) for a in (proc.map_ids, proc.map_masses, proc.map_widths,
                                                                      proc.d1, proc.d2, proc.has_children))
        L.c_whizard_fill_mapping(i(c + 1), p(ids), p(m), p(w))
        L.c_whizard_fill_tree_structure(i(c + 1), p(d1), p(d2), p(hc), p(np.zeros(proc.n_prt, np.int32)))
    L.c_whizard_init_gpu_phs()
    assert L.gpu_phs_last_error() == 0, L.gpu_phs_last_error_message()
    L.c_whizard_init_channel_ids(i(n), i(nc), (ctypes.c_int * nc)(*np.cumsum(counts).tolist()))
    e = np.full(n, proc.sqrts / 2)
    x, factors, volumes, oks = np.full((n, proc.n_x), 0.5), np.zeros(n * nc), np.zeros(n), np.zeros(n, np.bool_)
    mom, x_out, boost = np.zeros((n, proc.n_out, 4)), np.zeros(n * nc * proc.n_x), ctypes.c_bool(True)
    def call():
        L.c_whizard_gen_phs_from_x_gpu(p(e), p(e), ctypes.byref(boost), i(n), i(nc), i(proc.n_x), p(x), p(factors),
                                       p(volumes), p(oks), p(mom), p(x_out))
        return L.gpu_phs_last_error()
    return L, call
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("hip_host") / "libhip_host.so")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-I/opt/rocm/include",
                           os.path.join(HERE, "hip_host.cpp"), "-o", lib])

    def run(body):
        script = PRELUDE.format(runtime=lib, root=ROOT, here=HERE) + body
        r = subprocess.run([sys.executable, "-c", script], capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stdout + r.stderr
        return r.stdout
    return run


@pytest.mark.parametrize("events,wait", [(100_000, 0), (100_000, 5), (100_000, 9), (100_000, 12), (100_000, 15),
                                         (150_000, 12), (150_000, 20)])
def test_failed_host_call_leaves_no_copy_behind(run, events, wait):
    """A wait that fails in the middle of a host call (300,000 events: some 30 chunks, a ring of eight slots, two
    streams; 450,000: larger chunks on one) ends the call with an error and with no transfer in flight, so that the pinned slots may be
    released at once."""
    run(f"""
L, call = whizard(W.process_c1(), [{events}] * 3)
assert call() == 0
H.hip_host_fail_wait({wait})
assert call() != 0
pending = H.hip_host_pending()
L.c_whizard_finalize_gpu_phs()
assert H.hip_host_violations() == 0, "memory released under a copy"
assert pending == 0, pending
""")


def test_copy_threads_sleep_while_the_device_works(run):
    """The threads that copy between pinned and pageable memory wait asleep: a host call whose DMAs take 20 ms each
    (here the waits for them) takes next to no processor time."""
    run("""
L, call = whizard(W.process_c1(), [30_000] * 3)
assert call() == 0   # (starts the threads, touches the arrays)
H.hip_host_wait_us(20_000)
def used():
    r = resource.getrusage(resource.RUSAGE_SELF)
    return r.ru_utime + r.ru_stime
best = 1e9
for _ in range(4):   # (numpy's own threads may spin for a while after the start)
    cpu, wall = used(), time.perf_counter()
    assert call() == 0
    cpu, wall = used() - cpu, time.perf_counter() - wall
    assert wall > 0.15, wall
    best = min(best, cpu / wall)
assert best < 0.5, best
""")


def test_init_makes_the_streams_of_the_host_calls(run):
    """The streams of the host calls are made, and have had their first transfers, when c_whizard_init_gpu_phs
    returns, not in the first call for events; the program may end, or call again, at any time after it."""
    run("""
L, call = whizard(W.process_c1(), [100_000] * 3)
made = H.hip_host_streams()
assert made > 0 and H.hip_host_used_streams() == made
assert H.hip_host_pending() == 0
for _ in range(2):
    assert call() == 0
    assert H.hip_host_streams() == made
L.c_whizard_reset_generator()
assert call() == 0
L.c_whizard_finalize_gpu_phs()
assert H.hip_host_violations() == 0
""")


def test_grid_draw_asks_for_its_lds(run):
    """The draw's tables (464 bytes of LDS per random, and 544 for each wave) stay within the device's limit: where four
    waves do not fit, fewer draw."""
    run("""
H.hip_host_lds(65536)
for n_out in (8, 12):
    pl = plan(W.process_large(n_out), [100, 100])
    grid = G.Grid(pl._keep[0][0])
    launches()
    grid.generate(pl, 1, Stream)
    assert any("grid_generate" in k for k in launches())
assert 0 < H.hip_host_most_lds() <= 65536, H.hip_host_most_lds()
""")


@pytest.mark.parametrize("process,counts,beams,budgets", [
    ("W.process_c1()", [5000] * 3, False, {0}),                # three shapes of a group in one launch
    ("W.process_shapes(5)", [300] * 42, False, {0}),
    ("W.process_c1()", [5000, 0, 0], False, {0, 5}),           # one shape of four particles: its own kernels
    ("W.process_c1()", [5000, 0, 0], True, {0}),               # with per-event beams it has one budget
    ("W.process_friends(4)", [5000] * 4, False, {0, 3, 4}),    # the generic kernel
])
def test_autotuner_tries_the_budgets_that_select_a_kernel(run, process, counts, beams, budgets):
    """Launches that ignore waves_per_eu are not timed under several values of it: each is as fast as the others, and
    the one left in place (here every later candidate looks faster) would mean something to other launches."""
    run(f"""
proc = {process}
pl = plan(proc, ({counts} + [0] * proc.n_channels)[:proc.n_channels])
if {beams}:
    for k, (_, buf) in enumerate(pl._keep):
        e = Array(buf.x.shape[0])
        e.a[:] = proc.sqrts / 2
        pl.set_event_beams(k, e, e)
H.hip_host_elapsed(30.0, 0.001)
report = pl.autotune(stream=Stream, reps=1)
tried = [k.split(":")[1].split("/") for k in report.split(";")[-1].split()]
assert len(tried) > 5
assert {{int(t[3]) for t in tried if int(t[2]) == 0}} == {budgets}, report
""")


def test_plan_building_sorts_segments_not_tiles(run):
    """The tile table of 20 million events (78,000 tiles, 150 segments of four processes) is built in less time than
    numpy takes to sort as many random numbers stably."""
    run("""
class Events(Array):   # a segment's array that only an address is wanted of
    def __init__(self, *shape):
        self.shape, self.dtype = shape, np.float64
    def data_ptr(self):
        return 1 << 20

segs = []
for proc in (W.process_c0(), W.process_c1(), W.process_c2(), W.process_2to6()):
    ph = G.ProcessHandle(proc)
    for c in range(proc.n_channels):
        n = 2 * 5_000_000 * (c + 1) // (proc.n_channels * (proc.n_channels + 1))
        segs.append((ph, c, G.EventBuffers(Events(n, proc.n_x), Events(n, proc.n_out, 4), Events(n), Events(n), Events(n))))
def fastest(f):
    t = []
    for _ in range(9):
        start = time.perf_counter()
        f()
        t.append(time.perf_counter() - start)
    return min(t)
tiles = G.Plan(segs).info()["n_tiles"]
numbers = np.random.default_rng(1).random(tiles)
build, sort = fastest(lambda: G.Plan(segs).close()), fastest(lambda: np.argsort(numbers, kind="stable"))
assert tiles > 70_000
assert build < sort, (build, sort)
""")


@pytest.mark.parametrize("order", [0, 1])
def test_small_shapes_share_one_generic_launch(run, order):
    """Where a launch shape has no kernels for groups of shapes (a persistent grid), the small shapes of a tile class
    run in one launch of the generic kernel, whatever their numbers of particles, and every large one in its own; else
    each group in one of its own."""
    run(f"""
segs, large = [], 0
for n_out in (5, 6):
    ph = G.ProcessHandle(W.process_shapes(n_out, 1))
    for c in range(ph.proc.n_channels):
        n = 140 if c % 3 == 0 else 70
        large += n == 140
        segs.append((ph, c, G.EventBuffers(Array((n, ph.n_x)), Array((n, n_out, 4)), Array(n), Array(n),
                                           Array(n, np.uint8))))
pl = G.Plan(segs)
pl.set_config(block=64, ept=1, order={order})
pl.set_merge_below(100)
for grid in (0, 256, 0, 256):
    pl.set_config(grid=grid)
    launches()
    pl.run(Stream)
    names = launches()
    if grid:
        assert len(names) == large + 1 and sum("ELin1E" in k for k in names) == 1, names
    else:
        assert len(names) == 2 and all("forward_shapes_kernel" in k for k in names), names
""")


def test_inverse_tables_are_cheap(run):
    """Preparing the inverse of a process (2,000 channels of eight particles) takes a small part of the time that
    compiling its trees takes, and a call with other output rows prepares nothing again."""
    run("""
proc = W.process_large(8, 2000)
ph, L = G.ProcessHandle(proc), G.lib()
buf = Array((64, 8))
one = [(ph, 0, G.EventBuffers(Array((64, proc.n_x)), Array((64, 8, 4)), Array(64), Array(64), Array(64, np.uint8)))]
def seconds(f):
    start = time.perf_counter()
    f()
    return time.perf_counter() - start
def inverse(pl, row):
    rows = np.array([row], np.int64)
    assert L.gpu_phs_plan_inverse(pl.handle, p(rows), 1000, p(buf.a), p(buf.a), 0, None) == 0
compiled = min(seconds(lambda: G.ProcessHandle(proc).close()) for _ in range(7))
first, again = [], []
for _ in range(7):
    pl = G.Plan(one)
    first.append(seconds(lambda: inverse(pl, 0)))
    again += [seconds(lambda: inverse(pl, row)) for row in (1, 2, 3)]
assert min(first) < 0.1 * compiled, (min(first), compiled)
assert min(again) < 0.1 * min(first), (min(again), min(first))
""")


@pytest.mark.parametrize("process", ["W.process_c1()", "W.process_2to6()", "W.process_large(8)", "W.process_friends(6)"])
def test_launches_have_no_empty_workgroups(run, process):
    """A plan of many segments shorter than a tile launches workgroups for the events there are, not for those its
    tiles have room for: forward, plain and inverse, at every number of sub-tiles per tile."""
    run(f"""
proc = {process}
ph, segs = G.ProcessHandle(proc), []
for k in range(300):
    n = (70, 64, 1, 129)[k % 4]
    segs.append((ph, k % proc.n_channels, G.EventBuffers(Array((n, proc.n_x)), Array((n, proc.n_out, 4)), Array(n), Array(n),
                                                         Array(n, np.uint8))))
used = 75 * (2 + 1 + 1 + 3)   # workgroups of 64 events
rows = np.zeros(300, np.int64)
pl = G.Plan(segs)
for ept in (1, 4, 16, 2):
    pl.set_config(block=64, ept=ept, grid=0)
    H.hip_host_groups()
    pl.run(Stream)
    assert used <= H.hip_host_groups() <= 1.2 * used, ept
    pl.run_plain(Stream)
    assert used <= H.hip_host_groups() <= 1.2 * used, ept
    if not proc.friends_or_zero().any():
        assert G.lib().gpu_phs_plan_inverse(pl.handle, p(rows), 1000, p(rows), p(rows), 64, None) == 0
        n = H.hip_host_groups()
        assert n % used == 0 and n // used <= proc.n_channels, (ept, n)
pl.set_config(ept=16, grid=100)   # a persistent grid goes through tiles
pl.run(Stream)
assert H.hip_host_groups() <= 400
""")


@pytest.mark.parametrize("process", ["W.process_c1()", "W.process_2to6()", "W.process_friends(6)"])
def test_tables_are_not_written_under_queued_launches(run, process):
    """A plan's tables are written over only when what is queued on a stream of its own (which no copy waits for)
    has run: other launch shapes, beams and orders, other output rows of the inverse, other buffers of the
    adjoint, other weights of a grid."""
    run(f"""
proc, L = {process}, G.lib()
n = proc.n_channels
pl = plan(proc, [200] * n)
stream = ctypes.c_void_p()
assert H.hipStreamCreateWithFlags(ctypes.byref(stream), 1) == 0
class Own:
    cuda_stream = stream.value
def quiet(what, change):
    # a launch, the change, and a launch again
    pl.run(Own)
    change()
    pl.run(Own)
    assert H.hip_host_overwritten() == 0, what
quiet("nothing", lambda: None)
for config in (dict(grid=256), dict(grid=0), dict(block=64), dict(ept=4), dict(order=1)):
    quiet(config, lambda: pl.set_config(**config))
quiet("merge_below", lambda: L.gpu_phs_plan_set_merge_below(pl.handle, 0))
beams = Array(200)
quiet("beams", lambda: L.gpu_phs_plan_set_event_beams(pl.handle, 0, p(beams.a), p(beams.a)))
quiet("beams off", lambda: L.gpu_phs_plan_set_event_beams(pl.handle, 0, None, None))
buf = Array(64)
for row in (0, 1, 2, 2):
    rows = np.arange(n, dtype=np.int64) * 200 + row
    assert L.gpu_phs_plan_inverse(pl.handle, p(rows), 10 ** 6, p(buf.a), p(buf.a), 0, stream) == 0
    assert H.hip_host_overwritten() == 0, ("inverse", row)
for _ in range(3):
    keep = [Array((200, proc.n_x)) for _ in range(n)]
    adj = (G._AdjSegment * n)(*(G._AdjSegment(None, None, k.data_ptr(), None) for k in keep))
    assert L.gpu_phs_plan_adjoint(pl.handle, adj, 0, 0, p(buf.a), stream) == 0
    assert H.hip_host_overwritten() == 0, "adjoint"
grid = L.gpu_phs_grid_create(pl._keep[0][0].handle)
for seed in range(3):
    assert L.gpu_phs_grid_generate(grid, pl.handle, ctypes.c_uint64(seed), stream) == 0
    assert H.hip_host_overwritten() == 0, "grid"
""")
