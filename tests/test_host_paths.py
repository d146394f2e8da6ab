"""What the library does on the host, checked with no GPU: liberod.so runs over
a stand-in for the HIP runtime (hip_double.cpp) that keeps memory on the host
and logs allocations, copies and launches.  Each test is a short program in a
process of its own."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "elasticapp_amd", "liberod.so")

PRELUDE = """
import ctypes, re, sys
import numpy as np
import elasticapp_amd as ea
from elasticapp_amd import FP32_BULK, FP64, DeviceBlock
D = ctypes.CDLL(sys.argv[1])
D.double_log.restype = ctypes.c_char_p
D.double_live.restype = ctypes.c_size_t

def log(word=""):
    return [l for l in D.double_log().decode().splitlines() if word in l]

def launches():
    # (precision, elements per thread, threads, pieces, tiles, steps) of every fused launch
    return [(a[0], int(a[1]), int(a[2]), int(a[3]), int(a[4]), int(a[5])) for a in
            re.findall(r"k_fusedI([df])Li(\\d+)ELi(\\d+)ELi\\d+ELb([01])E\\S* grid (\\d+) steps (\\d+)", D.double_log().decode())]

def fast(name, faster=b""):
    D.double_fast(name, faster)

def block(lengths):
    b = DeviceBlock(list(lengths))
    b.set_rod_dt(1e-5)
    D.double_clear()
    return b
"""


@pytest.fixture(scope="session")
def run(tmp_path_factory):
    if not os.path.exists(LIB):
        if not os.path.exists("/opt/rocm/bin/hipcc"):
            pytest.skip("liberod.so not built and no hipcc here")
        from elasticapp_amd import build
        build.build()
    so = str(tmp_path_factory.mktemp("hip") / "hip_double.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-shared", "-fPIC", "-o", so,
                    os.path.join(ROOT, "tests", "hip_double.cpp")], check=True)

    def go(program):
        env = dict(os.environ)
        env["LD_PRELOAD"] = " ".join([so] + env.get("LD_PRELOAD", "").split())
        r = subprocess.run([sys.executable, "-c", PRELUDE + program, so], cwd=ROOT, env=env, capture_output=True, text=True,
                           timeout=120)
        assert r.returncode == 0, r.stdout + r.stderr
        return r.stdout

    return go


def test_memory_made_on_first_use_is_on_the_batchs_device(run):
    """A program may make another device current between two calls on a batch:
    what the calls allocate, and the events they record, are the batch's
    device's, and the program's device is current again afterwards."""
    run("""
blk = block([400, 30])            # on device 0
D.double_set_device(1)
blk.step(1e-5, 30)                # second copy of the state
blk.get_field("Position")         # pinned stage
blk.step_fused(20, FP64)          # pieces: second copy, plan
assert log("k_steps") and any(l[3] for l in launches())
assert all(l.endswith("foreign 0") for l in log("foreign")), log("foreign")
big = block([70000])              # on device 1
D.double_set_device(0)
big.get_field("Director")         # ring and events
big.autotune(FP32_BULK, 4)
assert len(launches()) > 1
assert all(l.endswith("foreign 0") for l in log("foreign")), log("foreign")
d = ctypes.c_int()
assert D.hipGetDevice(ctypes.byref(d)) == 0 and d.value == 0
assert D.double_live(0) > 0 and D.double_live(1) > 0
blk.close(); big.close()
assert D.double_live(0) == 0 and D.double_live(1) == 0
""")


@pytest.mark.parametrize("halo,pieces", [(2, 0), (3, 0), (5, 0), (6, 1), (8, 1), (16, 1), (32, 1)])
def test_small_fp64_batches_with_a_short_halo(run, halo, pieces):
    """FP64 rods of 257 to 512 elements take pieces of 256 lanes only with a halo
    whose launches pay for them; with a shorter one they run whole, in 512, a
    call in one launch.  Calls of fewer than 16 steps run whole with any."""
    run("""
blk = block([300, 400, 20])
blk.set_fused_pieces(0, 0, %d)
blk.step_fused(100, FP64)
assert any(l[3] for l in launches()) == %d and {l[1:3] for l in launches()} == {(1, 256 if %d else 512)}, launches()
assert %d or len(launches()) == 1
D.double_clear()
blk.step_fused(15, FP64)
assert [l[1:4] for l in launches()] == [(1, 512, 0)]
""" % (halo, pieces, pieces, pieces))


@pytest.mark.parametrize("lengths", ["[300, 400, 20]", "[3, 301] + [10] * 59", "[512] + [2] * 200"])
def test_small_fp64_batches_need_one_queue(run, lengths):
    """Rods that need no cut beside FP64 rods of 257 to 512 elements are no group
    of their own: two groups run side by side only where the runtime gives the
    batch's two streams two hardware queues, and take their sum elsewhere."""
    run("""
blk = block(%s)
blk.step_fused(100, FP64)
steps = [l[5] for l in launches()]
assert {l[3] for l in launches()} == {1} and sum(steps) == 100, launches()
assert blk.fused_config()[:2] == (256, 1) and blk.fused_pieces()[0] == 256
assert blk.fused_pieces()[4] == sum(max(2, -(-n // 128)) for n in blk.n_elems if n > 256)  # (halos of 64)
""" % lengths)


@pytest.mark.parametrize("halo,pieces", [(0, 1), (96, 1), (97, 0), (100, 0), (127, 0), (128, 0), (200, 0)])
def test_small_fp64_batches_with_a_long_halo(run, halo, pieces):
    """FP64 rods of 257 to 512 elements take pieces of 256 lanes only with a halo
    that leaves them room; with a longer one they run whole, in 512."""
    run("""
blk = block([300, 400, 20])
blk.set_fused_pieces(0, 0, %d)
blk.set_fused_config(0, 0, 200)
blk.step_fused(200, FP64)
assert all(l[:3] == (("d", 1, 256) if %d else ("d", 1, 512)) for l in launches()), launches()
assert any(l[3] for l in launches()) == %d
""" % (halo, pieces, pieces))


def test_short_fp64_calls_keep_small_batches_whole(run):
    """Pieces cost a launch two passes over the state more: a call whose launches
    are shorter than a halo runs rods of 257 to 512 elements whole, also between
    longer calls, and each kind's plan is made once."""
    run("""
blk = block([300, 400, 270])
def pieces(n, graph=0):
    D.double_clear()
    blk.step_fused_graph(n, graph, FP64) if graph else blk.step_fused(n, FP64)
    ls = launches()
    assert ls and len({l[3] for l in ls}) == 1
    return ls[0][3]
assert [pieces(n) for n in (1, 8, 15)] == [0, 0, 0]
assert len(launches()) == 1 and not log("k_copy_cut_state")
assert [pieces(n) for n in (16, 100, 5, 200)] == [1, 1, 0, 1]
for n, p in ((8, 0), (64, 1), (8, 0)):
    assert pieces(n) == p and not log("copy device")  # (no plan goes up again)
assert pieces(90, 8) == 0 and pieces(90, 30) == 1 and pieces(8, 30) == 0
blk.step_fused_graph(90, 30, FP64)
assert len(log("replay")) == 3 and not log("capture")  # (the graph of 30 steps is still that plan's)
blk.set_fused_config(0, 0, 8)
assert pieces(100) == 0
""")


@pytest.mark.parametrize("precision", ["FP64", "FP32_BULK"])
def test_a_pool_stays_within_its_hbm_budget(run, precision):
    """What a server allocates for rods of 257 to 512 elements, from its first
    request to the last, is what it reports."""
    run("""
lib = block([300, 400, 270, 500])
before = D.double_live(0)
srv = ea.Server(lib, [(512, 400)], %s, 20)
for i in range(6):
    srv.submit(i, [0, 1, 2, 3][: 1 + i %% 4], 40)
done = []
while len(done) < 6:
    done += srv.tick()
used, said = D.double_live(0) - before, srv.status()["pool_bytes"]
assert used <= 1.02 * said, (used, said)  # (tables of a few KB beside the fields)
assert launches() and not any(l[3] for l in launches())
""" % precision)


def test_a_tuned_plan_outlives_calls_of_another_length(run):
    """The plan an autotune leaves in place stands for calls longer and shorter
    than its trials, also where the caller had requested another shape."""
    run("""
for precision, name in ((FP32_BULK, b"k_fusedIfLi1ELi256E"), (FP64, b"k_fusedIdLi1ELi256E")):
    for lanes in (0, 512):
        blk = block([200, 250, 30, 100])
        blk.set_fused_config(lanes, 0, 0)
        fast(name)
        blk.autotune(precision, 4)
        for n in (100, 3, 100):
            D.double_clear()
            blk.step_fused(n, precision)
            assert [l[1:3] for l in launches()] == [(1, 256)], (precision, lanes, n, launches())
""")


@pytest.mark.parametrize("lengths", ["[2500] * 12 + [6000] * 12", "[1100, 1500]", "[700] * 40 + [5000] * 3", "[1300, 30, 200, 2000]",
                                     "[5000] * 40", "[400, 100, 512]"])
@pytest.mark.parametrize("precision,letter", [("FP64", "d"), ("FP32_BULK", "f")])
def test_the_autotuner_keeps_the_plan_it_timed(run, precision, letter, lengths):
    """Whichever shape is fastest: the launches of the batch afterwards are the
    ones its trial timed, in their number, pieces and steps, after replans too,
    and cover the plan of an untuned batch."""
    run("""
T = 60
free = block(%(lengths)s)
free.step_fused(T, %(precision)s)
free = launches()
trials = []
for shape in ("Li1ELi256E", "Li1ELi512E", "Li2ELi512E", "Li2ELi256E"):
    blk = block(%(lengths)s)
    fast(("k_fusedI%(letter)s" + shape).encode())
    best = blk.autotune(%(precision)s, T)
    seen = launches()
    trials += seen
    for replan in (0, 1, 2):
        D.double_clear()
        if replan == 1:
            blk.set_fused_split(*blk.fused_split()[:2])
        if replan == 2:
            assert abs(blk.autotune(%(precision)s, T) - best) < 1e-6, shape
            D.double_clear()
        blk.step_fused(T, %(precision)s)
        now = launches()
        n = len(now)
        assert any(seen[i:i + n] == now for i in range(len(seen))), (shape, replan, now)
        assert abs(blk.last_kernel_ms()[0] / T - best) < 1e-6, (shape, replan)
n = len(free)
assert any(trials[i:i + n] == free for i in range(len(trials))), free
""" % dict(precision=precision, letter=letter, lengths=lengths))


@pytest.mark.parametrize("lengths,whole", [("[105, 258, 130, 200] * 3", 1), ("[40] * 20 + [10]", 1), ("[3, 512]", 1),
                                           ("[3, 513]", 0), ("[700] * 4 + [5000] * 3", 0)])
def test_a_tuned_fp32_batch_keeps_its_rods_whole(run, lengths, whole):
    """FP32-bulk rounds a rod that is cut by its halo, so where 512 lanes hold
    every rod none is cut, of whatever shape the trials were fastest.  A caller
    that asks for pieces has them, and FP64, the same bits either way, has any."""
    run("""
T, cut = 60, set()
def tuned(precision, shape, lanes=0):
    blk = block(%(lengths)s)
    blk.set_fused_pieces(lanes, 0, 0)
    fast(shape)
    blk.autotune(precision, T)
    D.double_clear()
    blk.step_fused(T, precision)
    return any(l[3] for l in launches())
for shape in (b"Li1ELi64E", b"Li1ELi128E", b"Li1ELi256E", b"Li1ELi512E", b"Li2ELi64E", b"Li2ELi256E", b"Li2ELi512E"):
    cut.add(tuned(FP32_BULK, b"k_fusedIf" + shape))
assert (cut == {False}) == %(whole)d, cut
if max(block(%(lengths)s).n_elems) > 64:
    assert tuned(FP32_BULK, b"k_fusedIfLi1ELi64E", 64)
    assert tuned(FP64, b"k_fusedIdLi1ELi64E")
""" % dict(lengths=lengths, whole=whole))


def test_fp64_on_a_batch_tuned_for_fp32(run):
    """FP64 has no registers for two elements per thread in one wave: it takes
    128 lanes at one where the autotuner chose that shape for FP32-bulk, as the
    main one or the second group's, and a caller's own request stands."""
    run("""
def shapes(b, precision):
    D.double_clear()
    b.step_fused(30, precision)
    return {l[1:3] for l in launches()}
blk = block([100] * 50)
fast(b"k_fusedIfLi2ELi64E")
blk.autotune(FP32_BULK, 20)
for _ in range(2):
    assert shapes(blk, FP32_BULK) == {(2, 64)} and shapes(blk, FP64) == {(1, 128)}
    assert not _ or not log("copy device")  # (both plans are kept)
blk.set_fused_config(128, 2, 0)
assert shapes(blk, FP64) == {(2, 64)}

fast(b"k_fusedIfLi1ELi512E", b"k_fusedIfLi2ELi64ELi0ELb0E")
blk = block([500] * 300 + [20] * 300)
blk.autotune(FP32_BULK, 20)
assert blk.fused_split()[:2] == (128, 2)
for _ in range(2):
    assert shapes(blk, FP32_BULK) == {(1, 512), (2, 64)} and shapes(blk, FP64) == {(1, 512), (1, 128)}
    assert not _ or not log("copy device")
blk = block([500] * 300 + [20] * 300)
blk.set_fused_split(128, 2)
assert (2, 64) in shapes(blk, FP64)
""")


def test_fp32_on_a_batch_tuned_for_fp64(run):
    """FP32-bulk rounds a rod that runs as a piece by its halo: which rods do is
    the same whether the FP64 call that made the plan came before or after."""
    run("""
def tuned():
    blk = block([300, 400, 20, 250])
    fast(b"k_fusedIdLi1ELi256E")
    blk.autotune(FP64, 100)
    return blk
def plan(blk, precision):
    D.double_clear()
    blk.step_fused(100, precision)
    return sorted(set(l[1:5] for l in launches()))
blk = tuned()
blk.set_fused_split(0, 0)          # (plans are made anew)
first = plan(blk, FP32_BULK)
assert {l[2] for l in first} == {0, 1}, first
both = plan(blk, FP64)
assert {l[2] for l in both} == {1}, both
blk = tuned()
for _ in range(2):
    assert plan(blk, FP64) == both and plan(blk, FP32_BULK) == first
    assert not _ or not log("copy device")  # (both plans are kept)
""")


def test_a_requested_halo_is_not_widened(run):
    """A halo of 16 that the caller asked for stays 16, in any precision and
    after an autotune; one left free widens, and is free again with 0."""
    run("""
for precision, name in ((FP64, b"k_fusedIdLi1ELi256E"), (FP32_BULK, b"k_fusedIfLi1ELi256E")):
    fast(name)
    for tuned in (0, 1):
        blk = block([1500, 2000])
        counts = []
        for halo in (0, 16, 0):
            blk.set_fused_pieces(0, 0, halo)
            if tuned:
                blk.autotune(precision, 64)
            D.double_clear()
            blk.step_fused(64, precision)
            counts.append((max(l[5] for l in launches()), blk.fused_pieces()[4]))
        assert [c[0] for c in counts] == [64, 16, 64], counts
        assert counts[0] == counts[2] and counts[0][1] > counts[1][1], counts
""")


@pytest.mark.parametrize("n", ["25", "26", "101", "2**31 + 5", "2**40 + 7", "2**62 + 3"])
def test_launches_of_any_number_of_steps(run, n):
    """However many op-by-op steps one call asks for, each launch takes 12 of
    them at most and fits its workgroups."""
    run("""
blk = block([400, 30])
D.double_fail_after(ctypes.c_long(100))
try:
    blk.step(1e-9, %(n)s)
except ea.ErodError:
    pass
steps = [tuple(int(x) for x in re.search(r"steps (-?\\d+) left (-?\\d+) own (-?\\d+)", l).groups()) for l in log("k_steps")]
assert steps and all(1 <= s <= 12 and left == s and own == 255 - 2 * s for s, left, own in steps), steps
assert len(steps) %% 2 == 0 and (len(steps) == 100 or sum(s[0] for s in steps) == %(n)s - 1), steps
""" % dict(n=n))


@pytest.mark.parametrize("room,several", [(1 << 20, False), (4 << 20, False), (10 << 20, False), (64 << 20, True)])
def test_op_by_op_steps_leave_memory_to_others(run, room, several):
    """The second copy of the state is taken where the device has plenty of room
    for it; otherwise every step goes call by call, and nothing is kept."""
    run("""
blk = block([40000, 30])           # a copy of 5.8 MB
before = D.double_live(0)
D.double_capacity(ctypes.c_size_t(before + %d))
blk.step(1e-5, 5)
assert bool(log("k_steps")) == %s
assert len(log("k_kinematic")) == (2 if %s else 10)
assert (D.double_live(0) > before) == %s
""" % (room, several, several, several))
