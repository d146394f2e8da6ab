"""Several op-by-op steps in one launch: `step(n)` takes its first n - 1 steps
without writing the derived fields, several per launch, one workgroup per run
of slots with recomputed slots beside it.  Every field of the block, ghosts
included, equals the stepper's calls issued one by one, bitwise, at block
sizes around a workgroup's 256 slots, at step counts around the launch split,
and with every hook; the state equals the oracle's bitwise."""
import numpy as np
import pytest

from elasticapp_amd import FIELDS
from tests.gpu_helpers import STATE, device_block, oracle_system, random_workload

pytestmark = pytest.mark.gpu


def _workload(lengths, hooks):
    wl = random_workload(0, 0, 0, seed=sum(lengths) + 5, forces=hooks != "none", lengths=list(lengths))
    if hooks == "all":
        for r, n in enumerate(wl.n_elems):
            st = wl.states[r]
            i = (0, n, n // 2)[r % 3]
            wl.clamps.append((r, st["Position"][:, i].copy(), st["Director"][:, min(i, n - 1)].copy(), i))
            if r % 2:
                wl.forces[r] = (r, wl.forces[r][1], 1 + r % 2, 2 * wl.dt, 7 * wl.dt)
        wl.gravity = (0.1, 0.0, -9.81)
        z = float(np.median([st["Position"][2].min() for st in wl.states]))
        wl.contact = (1e3, 10.0, 0.3, 10.0, z, 0.01, (0.0, 0.6, 0.8))
    return wl


def _calls(blk, dt, n):
    t = 0.0
    for _ in range(n):
        blk.kinematic_update(dt)
        t += 0.5 * dt
        blk.apply_post_kinematic(t)
        blk.compute_internal_dynamics(t)
        blk.apply_pre_dynamic(t)
        blk.dynamic_update(dt)
        blk.apply_post_dynamic(t)
        t += 0.5 * dt
        blk.kinematic_update(dt)


# lengths: slots (elements + ghosts + the last node) just under, at and over one
# workgroup, rod ends at and around its edges, and many workgroups
@pytest.mark.parametrize("lengths", [(2,), (255,), (256,), (120, 133), (120, 134), (3, 249, 2, 5), (700,),
                                     (236, 2, 2, 238, 2, 240, 31), (64,) * 40])
@pytest.mark.parametrize("hooks", ["none", "all"])
def test_step_equals_its_calls(lengths, hooks):
    wl = _workload(lengths, hooks)
    a, b = device_block(wl), device_block(wl)
    sysm = oracle_system(wl, variant="devmath")
    # 1 and 2: no launch of several steps (or one, in place); 3: one step per
    # launch; then uneven and even splits over two and more launches
    for n in (1, 2, 3, 10, 17, 18, 34):
        _restart(a, wl)
        _restart(b, wl)
        a.step(wl.dt, n)
        _calls(b, wl.dt, n)
        for tag in FIELDS:
            assert np.array_equal(a.get_field(tag), b.get_field(tag), equal_nan=True), (tag, n)
    sysm.step(wl.dt, 34)
    for r in range(len(wl.n_elems)):
        for tag in STATE:
            assert np.array_equal(a.get_rod(tag, r), sysm.rod_field(r, tag)), (tag, r)


def _restart(blk, wl):
    """The workload's state back into the block, at time 0."""
    blk.time = 0.0
    for r, st in enumerate(wl.states):
        for tag in STATE:
            blk.set_rod(tag, r, st[tag])


def test_undamped_block():
    wl = _workload((90, 300), "none")
    for st in wl.states:
        del st["ForceDampingRate"], st["TorqueDampingRate"]
    a, b = device_block(wl, damped=False), device_block(wl, damped=False)
    a.step(wl.dt, 20)
    _calls(b, wl.dt, 20)
    for tag in FIELDS:
        assert np.array_equal(a.get_field(tag), b.get_field(tag), equal_nan=True), tag
