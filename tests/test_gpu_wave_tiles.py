"""Tiles of one wave exchange neighbours' values between its lanes: bitwise the
results of a tile of several waves, for rods that end on a wave's last lane, beside it and across it, tiles with idle lanes, rods
of other directions in one wave, every environment, clamps at both ends, step
budgets, and (FP64) a rod of no numbers beside the others."""
import numpy as np
import pytest
import torch

from elasticapp_amd import FP32_BULK, FP64, DeviceBlock, assemble
from elasticapp_amd.workloads import UniformRods, build_block
from tests.gpu_helpers import STATE, random_workload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [FP64, FP32_BULK])
@pytest.mark.parametrize("env", ["none", "level", "tilted"])
@pytest.mark.parametrize("lanes,epl", [(64, 1), (128, 1), (512, 1), (128, 2)])
def test_tiles_of_one_wave(lanes, epl, env, precision):
    fits = [n for n in (63, 65, 126, 127, 128, 129, 191, 256, 257, 512) if n <= lanes]
    wl = random_workload(0, 0, 0, seed=700 + lanes, lengths=[2, 3, 62, 64, 31, 33, 2, 2] + fits)
    n = wl.n_elems[3]
    for r, i in ((0, 0), (3, 0), (3, n)):
        st = wl.states[r]
        wl.clamps.append((r, st["Position"][:, i].copy(), st["Director"][:, min(i, wl.n_elems[r] - 1)].copy(), i))
    if env != "none":
        wl.gravity = (0.0, 0.0, -9.81)
        # (rods lie on both sides of the plane)
        wl.contact = (1e2, 1.0, 0.3, 1.0, 0.0, 0.01) + (((0.0, 0.6, 0.8),) if env == "tilted" else ())
    wave, ref = build_block(wl), build_block(wl)
    wave.set_fused_config(lanes, epl, 0)
    ref.set_fused_config(1024, 2, 0)
    for steps in (1, 2, 30):
        for b in (wave, ref):
            if steps == 30:
                b.set_step_budget(1, 7)
                if precision == FP64:
                    v = b.get_rod("Velocity", 2)
                    v[:, 5] = np.nan
                    b.set_rod("Velocity", 2, v)
            b.step_fused(steps, precision)
        # (a spent budget leaves the plan to be made again)
        assert steps == 30 or wave.fused_config()[:2] == (lanes, epl)
        for r in range(len(wl.n_elems)):
            # (past the first NaN only the other rods, which must not see it)
            if r == 2 and steps == 30 and precision == FP64:
                continue
            for tag in STATE:
                a, b = wave.get_rod(tag, r), ref.get_rod(tag, r)
                assert np.isfinite(a).all() and np.array_equal(a, b), (steps, r, tag)


@pytest.mark.parametrize("precision", [FP64, FP32_BULK])
@pytest.mark.parametrize("n,per_cu,small,full", [(64, 640, (64, 1), (128, 2)), (100, 512, (128, 1), (128, 2)),
                                                 (129, 1024, (256, 1), (512, 2))])
def test_free_shapes_of_batches_that_fill_the_device(n, per_cu, small, full, precision):
    for more in (0, 1):
        count = per_cu * torch.cuda.get_device_properties(0).multi_processor_count // n + more
        st = random_workload(0, 0, 0, seed=800 + n, lengths=[n]).states[0]
        offsets = np.random.default_rng(n).normal(size=(count, 3))
        kappa = np.repeat(st["ReferenceCurvature"][None], count, axis=0)
        blk, ref = DeviceBlock([n] * count), DeviceBlock([n] * count)
        for b in (blk, ref):
            assemble(b, UniformRods(st, offsets, kappa))
            b.set_rod_dt(1e-5)
        ref.set_fused_config(1024, 2, 0)
        for b in (blk, ref):
            b.step_fused(3, precision)
        assert blk.fused_config()[:2] == (full if more and precision == FP32_BULK else small)
        assert all(np.array_equal(blk.get_field(t), ref.get_field(t)) for t in STATE)


@pytest.mark.parametrize("precision", [FP64, FP32_BULK])
@pytest.mark.parametrize("env", ["none", "tilted"])
@pytest.mark.parametrize("lanes,epl", [(64, 1), (128, 1), (256, 1), (512, 1), (128, 2), (512, 2), (1024, 2), (512, 4), (1024, 4)])
def test_a_rod_of_no_numbers_leaves_its_tile_alone(lanes, epl, env, precision):
    """Rods in one tile beside ones that went non-finite, at their ends or
    inside, in any part of their state, keep the bits they have without them."""
    wl = random_workload(0, 0, 0, seed=900 + lanes + epl, lengths=[7, 5, 9, 4, 11, 6, 13, 4, 5])
    if env == "tilted":
        wl.gravity = (0.0, 0.0, -9.81)
        wl.contact = (1e2, 1.0, 0.3, 1.0, 0.0, 0.01, (0.0, 0.6, 0.8))
    ref, blk = build_block(wl), build_block(wl)
    for b in (ref, blk):
        b.set_fused_config(lanes, epl, 0)
    lost = {0: ("Director", 0, np.nan), 2: ("Position", -1, np.inf), 4: ("Velocity", 0, np.nan),
            6: ("AngularVelocity", -1, -np.inf), 7: ("Position", 0, np.nan)}
    for r, (tag, i, value) in lost.items():
        a = blk.get_rod(tag, r)
        a[:, i] = value
        blk.set_rod(tag, r, a)
    for steps in (1, 1, 12):
        for b in (ref, blk):
            b.step_fused(steps, precision)
        for r in range(len(wl.n_elems)):
            if r not in lost:
                for tag in STATE:
                    assert np.array_equal(blk.get_rod(tag, r), ref.get_rod(tag, r)), (steps, r, tag)
    assert blk.fused_config()[:2] == (lanes, epl)
    assert [bool(f) for f in blk.check_finite()] == [r in lost for r in range(len(wl.n_elems))]
