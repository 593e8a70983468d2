"""Calls of the engine ABI whose work waits for a later one, checked on the CPU: the order in which
the engine launches, waits and copies, recorded by a HIP runtime that runs no kernel
(hip_recorder.c), and the memory it allocates.  Each case is a process of its own."""
import os
import subprocess
import sys

import pytest

from scenarios import ROOT

HEAD = r'''
import ctypes, re, sys, threading
GLOBAL, V, I = ctypes.RTLD_GLOBAL, ctypes.c_void_p, ctypes.c_int
rec = ctypes.CDLL(sys.argv[1] + "/hip_recorder.so", mode=GLOBAL)
lib = ctypes.CDLL(sys.argv[2] + "/alis_amd/libalis.so", mode=GLOBAL)
ec = ctypes.CDLL(sys.argv[1] + "/engine_client.so")
rec.hipRecLog.restype = lib.alis_dev_error.restype = ctypes.c_char_p
rec.hipRecOutside.restype = ctypes.c_long
rec.hipRecStreamOf.argtypes = [V]
ec.ec_world.restype = ec.ec_boxes.restype = ec.ec_beam.restype = ec.ec_device.restype = ec.ec_aux.restype = V
ec.ec_step.argtypes = ec.ec_aux.argtypes = ec.ec_commit_below.argtypes = [V, I]
ec.ec_device.argtypes = ec.ec_free.argtypes = ec.ec_disown.argtypes = [V]
lib.alis_dev_core.argtypes = lib.alis_dev_ghosts.argtypes = [V, I]
lib.alis_dev_batch_core.argtypes = lib.alis_dev_batch_post.argtypes = [V, I]
lib.alis_dev_strips.argtypes = [V, I, I]
lib.alis_dev_sync.argtypes = [V] + 6 * [I]
lib.alis_dev_synchronize.argtypes = lib.alis_dev_batch_release.argtypes = lib.alis_dev_release.argtypes = [V]
lib.alis_dev_batch_create.argtypes = [ctypes.POINTER(V), I, ctypes.POINTER(V)]
lib.alis_dev_batch_release.restype = lib.alis_dev_release.restype = None

def ok(rc):
    assert rc == 0, lib.alis_dev_error().decode()

def calls(f, *args):
    """(launch, kernel, half step of a curl, workgroups, stream) and (wait, stream, other) of f."""
    rec.hipRecClear()
    f(*args)
    out = []
    for line in rec.hipRecLog().decode().splitlines():
        what, name, n, s = line.split()
        if what == "wait":
            out.append((what, int(n), int(s)))
        else:
            half = re.search(r"k_curl\w*?I[fd]Li(\d)", name)
            out.append((what, re.search(r"k_[a-z_]+", name).group(), int(half.group(1)) if half else -1, int(n), int(s)))
    return out

def kernels(log):
    return [c[1] for c in log if c[0] == "launch"]

def batch(devices):
    B = V()
    ok(lib.alis_dev_batch_create((V * len(devices))(*devices), len(devices), ctypes.byref(B)))
    return B
'''


@pytest.fixture(scope="module")
def libs(tmp_path_factory):
    out = tmp_path_factory.mktemp("recorder")
    for name in ("hip_recorder", "engine_client"):
        subprocess.run(["gcc", "-O1", "-std=gnu99", "-shared", "-fPIC", f"-I{ROOT / 'include'}", "-o", str(out / f"{name}.so"),
                        str(ROOT / "tests" / f"{name}.c"), "-lpthread"], check=True)
    return out


def run(libs, code, **env):
    r = subprocess.run([sys.executable, "-c", HEAD + code, str(libs), str(ROOT)], capture_output=True, text=True, timeout=120,
                       cwd=libs, env={**os.environ, **env})
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.parametrize("worlds", [2, 3])
def test_parts_of_a_world_as_entries_of_their_own(libs, worlds):
    """ALIS_BATCH_PAIRS=0: the parts of a Bloch world run side by side in one launch, so neither may make
    the ghost copies along z, which need the other's values and write both: all copies are left to
    the end of the half step, as they are where the core runs by itself."""
    run(libs, f"""
wl = ctypes.CDLL(sys.argv[2] + "/alis_amd/libalis_workloads.so")
wl.wl_create.restype = wl.wl_device_of.restype = V
wl.wl_step.argtypes = wl.wl_device_of.argtypes = [V, I]
c = wl.wl_create(b"kpoints", {worlds}, 32, 64)
wl.wl_step(c, 1)
B = batch([wl.wl_device_of(c, q) for q in range({worlds})])

def half(h, apart):
    ok(lib.alis_dev_batch_core(B, h))
    if apart:
        ok(lib.alis_dev_synchronize(wl.wl_device_of(c, 0)))
    ok(lib.alis_dev_batch_post(B, h))

for h in range(2):
    posts = [[k[3] for k in calls(half, h, apart) if k[1] == "k_post_batch"] for apart in (True, False)]
    assert posts[0] and posts[0] == posts[1], posts
lib.alis_dev_batch_release(B)
""", ALIS_BATCH_PAIRS="0")


@pytest.mark.parametrize("boxes", [0, 1])
def test_cores_of_their_own_before_a_batch_post(libs, boxes):
    """alis_dev_core of every world, then the post of their batch: the curls come before the end of the half
    step that they belong to."""
    run(libs, f"""
W = [V(ec.ec_world(40, {boxes}, 1)) for _ in range(2)]
for w in W:
    ec.ec_step(w, 1)
dev = [ec.ec_device(w) for w in W] + [ec.ec_aux(w, 0) for w in W if {boxes}]
B = batch(dev)

def half(h):
    for d in dev:
        ok(lib.alis_dev_core(d, h))
    ok(lib.alis_dev_batch_post(B, h))

for h in (0, 1, 0, 1):
    log = calls(half, h)
    curls = [n for n, c in enumerate(log) if c[2] == h and c[1].startswith("k_curl")]
    posts = [n for n, c in enumerate(log) if c[1] == "k_post_batch"]
    assert len(curls) == len(dev) and posts and curls[-1] < posts[0], log
lib.alis_dev_batch_release(B)
""")


def test_ends_of_their_own_after_a_batch_core(libs):
    """The core of a batch, then alis_dev_ghosts of each world: the curl comes before the end of either half
    step."""
    run(libs, """
W = [V(ec.ec_world(40, 0, 0)) for _ in range(2)]
for w in W:
    ec.ec_step(w, 1)
dev = [ec.ec_device(w) for w in W]
B = batch(dev)

def half(h):
    ok(lib.alis_dev_batch_core(B, h))
    for d in dev:
        ok(lib.alis_dev_ghosts(d, h))

for h in (0, 1, 0, 1):
    k = kernels(calls(half, h))
    assert k[0] == "k_curl_batch" and k.count("k_curl_batch") == 1 and "k_post" in k, k
lib.alis_dev_batch_release(B)
""")


@pytest.mark.parametrize("below", [0, 1, 3, 4, 5, 8, 11])
def test_object_box_below_the_grid(libs, below):
    """A dispersive object whose box starts under kMIN: its arrays, laid out along the grid's quads, hold
    every cell of the box."""
    run(libs, f"""
W = ec.ec_world(40, 0, 1)
ok(ec.ec_commit_below(W, {below}))
assert rec.hipRecOutside() == 0
""")


def test_main_world_without_its_auxiliary_world(libs):
    """The auxiliary world of a TF/SF box released before its main world, which steps on without strips."""
    run(libs, """
W = ec.ec_boxes(64, 1, 0, 25)
ec.ec_step(W, 2)
D, A = ec.ec_device(W), ec.ec_aux(W, 0)
ec.ec_disown(W)
lib.alis_dev_release(A)

def step():
    for h in range(2):
        ok(lib.alis_dev_core(D, h))
        ok(lib.alis_dev_ghosts(D, h))

for _ in range(2):
    assert [c[2] for c in calls(step) if c[1].startswith("k_curl")] == [0, 1]
lib.alis_dev_release(D)
""")


@pytest.mark.parametrize("calls_made", [1, 2])
def test_auxiliary_world_outlives_a_deferred_step(libs, calls_made):
    """ALIS_FUSE=force: an auxiliary world's H half step waits for its main world's fused step; where that
    world is released first, the half step is made all the same."""
    run(libs, f"""
W = ec.ec_world(40, 1, 0)
ec.ec_step(W, 2)
D, A = ec.ec_device(W), ec.ec_aux(W, 0)
ec.ec_disown(W)

def part():
    ok(lib.alis_dev_core(D, 0))
    ok(lib.alis_dev_core(A, 0)), ok(lib.alis_dev_ghosts(A, 0))
    ok(lib.alis_dev_ghosts(D, 0))
    ok(lib.alis_dev_core(D, 1))
    ok(lib.alis_dev_core(A, 1))
    if {calls_made} == 2:
        ok(lib.alis_dev_ghosts(A, 1))
    lib.alis_dev_release(D)
    if {calls_made} == 1:
        ok(lib.alis_dev_ghosts(A, 1))
    ok(lib.alis_dev_synchronize(A))

k = [c[2] for c in calls(part) if c[1].startswith("k_curl") and c[3] <= 4]     # (the small world's)
assert k == [0, 1], k

def step():
    for h in range(2):
        ok(lib.alis_dev_core(A, h)), ok(lib.alis_dev_ghosts(A, h))

assert [c[2] for c in calls(step) if c[1].startswith("k_curl")] == [0, 1]
lib.alis_dev_release(A)
""", ALIS_FUSE="force")


def test_timing_counts_a_waiting_core(libs):
    """alis_dev_timing_read after alis_dev_core: the launch that the call asked for is counted."""
    run(libs, """
W = ec.ec_world(40, 0, 0)
ec.ec_step(W, 1)
D = ec.ec_device(W)
lib.alis_dev_timing.argtypes = [V, I]
lib.alis_dev_timing_read.argtypes = [V, I, ctypes.POINTER(ctypes.c_double), ctypes.POINTER(ctypes.c_long)]
ok(lib.alis_dev_timing(D, 1))
for h in range(2):
    ok(lib.alis_dev_core(D, h))
    ms, n = ctypes.c_double(), ctypes.c_long()
    ok(lib.alis_dev_timing_read(D, h, ctypes.byref(ms), ctypes.byref(n)))
    assert n.value == 1 and ms.value > 0
    ok(lib.alis_dev_ghosts(D, h))
""")


def test_whole_syncs_on_two_devices(libs):
    """Worlds on two GPUs, synced from either of them as the current device: events and streams of one
    device together, the caller's device left as it was."""
    run(libs, """
dev = []
for d in range(2):
    ok(rec.hipSetDevice(d))
    W = ec.ec_world(40, 0, 1)
    ec.ec_step(W, 1)
    dev.append(ec.ec_device(W))
for current in (1, 0):
    ok(rec.hipSetDevice(current))
    for D in dev + dev:
        log = calls(lambda: ok(lib.alis_dev_sync(D, 0, -1, 0, -1, 0, -1)))
        assert "k_mirror" in kernels(log) and "k_pack" not in kernels(log), log
        now = I()
        ok(rec.hipGetDevice(ctypes.byref(now)))
        assert now.value == current
assert rec.hipRecForeign() == 0
""")


def test_commits_syncs_and_releases_beside_a_whole_sync(libs):
    """While one thread waits inside a whole sync, another commits, steps, syncs and releases a world."""
    run(libs, """
import time
A = ec.ec_world(64, 0, 1)
ec.ec_step(A, 1)
dA = ec.ec_device(A)
rec.hipRecHold()
first = threading.Thread(target=lambda: ok(lib.alis_dev_sync(dA, 0, -1, 0, -1, 0, -1)))
first.start()
while not rec.hipRecWaiting():
    time.sleep(0.01)

def other():
    B = V(ec.ec_world(40, 0, 1))
    ec.ec_step(B, 1)
    ok(lib.alis_dev_sync(ec.ec_device(B), 0, -1, 0, -1, 0, -1))
    ec.ec_free(B)

second = threading.Thread(target=other, daemon=True)
second.start()
second.join(20)
late = second.is_alive()
rec.hipRecLetGo()
first.join()
assert not late
""")


@pytest.mark.parametrize("sphere", [0, 1])
def test_worlds_one_after_another_share_the_staging(libs, sphere):
    """A program that solves one world after another pays for the pinned chunks of its whole syncs once;
    worlds that pass without a whole sync give them back."""
    run(libs, f"""
def solve(sync):
    W = V(ec.ec_world(64, 0, {sphere}))
    ec.ec_step(W, 1)
    if sync:
        ok(lib.alis_dev_sync(ec.ec_device(W), 0, -1, 0, -1, 0, -1))
    before = rec.hipRecPinned()
    ec.ec_free(W)
    return before

first = solve(True)
assert first > 0
for _ in range(3):
    assert solve(True) == first         # (allocated so far: nothing new)
for _ in range(2):
    solve(False)
assert rec.hipRecPinnedNow() == 0
assert solve(True) == 2 * first
""")


@pytest.mark.parametrize("percent", [25, 60])
def test_auxiliary_worlds_step_beside_the_curl(libs, percent):
    """Auxiliary worlds on streams of their own (two TF/SF boxes): the main world's curl is launched before its
    stream waits for them, and the launch that applies their strips after."""
    run(libs, f"""
W = ec.ec_boxes(64, 2, 0, {percent})
ec.ec_step(W, 2)
log = calls(ec.ec_step, W, 2)
main = max((c for c in log if c[0] == "launch" and c[1].startswith("k_curl")), key=lambda c: c[3])[4]
seen = []
for c in log:
    if c[0] == "wait" and c[1] == main:
        seen.append("w")
    elif c[0] == "launch" and c[4] == main:
        seen.append(c[1][2])
order = "".join(seen)
assert re.fullmatch("(c(w+)p)+", order) and order.count("c") == 4, order
""")


@pytest.mark.parametrize("shared", [False, True])
def test_core_runs_while_the_host_evaluates_waves(libs, shared):
    """A source with per-cell waves: the E core is launched at its call, before the host evaluates them for the
    end of the half step; without such waves, or once they have ended, it waits for that call."""
    run(libs, f"""
shared = {shared}
W = [V(ec.ec_beam(40, 4)) for _ in range(2)]
for w in W:
    ec.ec_step(w, 2)
dev = [ec.ec_device(w) for w in W]
B = batch(dev) if shared else None
curl = "k_curl_batch" if shared else "k_curl"
core = lambda h: ok(lib.alis_dev_batch_core(B, h) if shared else lib.alis_dev_core(dev[0], h))
end = lambda h: ok(lib.alis_dev_batch_post(B, h) if shared else lib.alis_dev_ghosts(dev[0], h))
for waves in (True, False):              # (the second step here records none)
    assert kernels(calls(core, 0)) == ([curl] if waves else [])
    assert (curl in kernels(calls(end, 0))) == (not waves)
    assert kernels(calls(core, 1)) == []
    assert curl in kernels(calls(end, 1))[0]
if shared:
    lib.alis_dev_batch_release(B)
""")


def test_strips_take_a_cell_per_thread(libs):
    """The strips of two TF/SF boxes of 14 x 28 x 28 cells at the end of the E half step: two components on
    each face, about 12500 cells, a wavefront (64 threads) to as many of them."""
    run(libs, """
W = ec.ec_boxes(64, 2, 0, 60)
ec.ec_step(W, 2)
log = calls(ec.ec_step, W, 1)
main = max((c for c in log if c[0] == "launch" and c[1].startswith("k_curl")), key=lambda c: c[3])[4]
post = [c[3] for c in log if c[0] == "launch" and c[4] == main and c[1].startswith("k_post")]
assert len(post) == 2 and post[0] >= 12500 * 0.9 / 64, post
""")


@pytest.mark.parametrize("shared", [False, True])
def test_objects_are_passed_over_once_a_step(libs, shared):
    """Objects of more than a workgroup per compute unit: the current update of an H half step runs with what the objects do before the next E curl, in one
    launch; apart from it only where a call in between reads the currents or changes E."""
    run(libs, f"""
shared = {shared}
W = [V(ec.ec_world(64, 0, 5)) for _ in range(2)]
for w in W:
    ec.ec_step(w, 2)
dev = [ec.ec_device(w) for w in W]
B = batch(dev) if shared else None
both = "k_objects_batch" if shared else "k_objects"           # (update and currents)
currents = "k_currents_batch" if shared else "k_currents"
core = lambda h: ok(lib.alis_dev_batch_core(B, h) if shared else lib.alis_dev_core(dev[0], h))
end = lambda h: ok(lib.alis_dev_batch_post(B, h) if shared else lib.alis_dev_ghosts(dev[0], h))
half = lambda h: (core(h), end(h))
objects = lambda k: [n for n in k if n in ("k_ade", both, currents)]
read = lambda d: ok(lib.alis_dev_read_field(V(d), 0, 0, 2, buf))
buf = (ctypes.c_double * 400000)()
lib.alis_dev_read_field.argtypes = [V, I, I, I, V]
half(0), half(1)
for between in ("nothing", "fields", "currents", "ghosts"):
    assert objects(kernels(calls(half, 0))) == [both], between
    assert objects(kernels(calls(half, 1))) == [], between
    if between == "fields":              # (the fields do not depend on it)
        assert objects(kernels(calls(read, dev[0]))) == []
    if between == "currents":
        assert objects(kernels(calls(lambda: ok(lib.alis_dev_sync(dev[0], 0, -1, 0, -1, 0, -1))))) == ["k_ade"]
        apart = objects(kernels(calls(half, 0)))
        assert apart == (["k_ade", currents] if shared else [currents])
        half(1)
    if between == "ghosts":              # E's ghost copies without a core
        k = objects(kernels(calls(end, 0)))
        assert k == ["k_ade"] * (2 if shared else 1), k
""")
