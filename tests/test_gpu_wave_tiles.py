"""Tiles of one element per thread exchange neighbours' values between the
lanes of a wave: bitwise the results of two elements per thread, for rods that
end on a wave's last lane, beside it and across it, tiles with idle lanes, rods
of other directions in one wave, every environment, clamps at both ends, step
budgets, and (FP64) a rod of no numbers beside the others."""
import numpy as np
import pytest

from elasticapp_amd import FP32_BULK, FP64
from elasticapp_amd.workloads import build_block
from tests.gpu_helpers import STATE, random_workload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [FP64, FP32_BULK])
@pytest.mark.parametrize("env", ["none", "level", "tilted"])
@pytest.mark.parametrize("lanes", [64, 128, 256, 512])
def test_one_element_per_thread(lanes, env, precision):
    fits = [n for n in (63, 65, 128, 129, 191, 256, 257, 512) if n <= lanes]
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
    wave.set_fused_config(lanes, 1, 0)
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
        assert steps == 30 or wave.fused_config()[:2] == (lanes, 1)
        for r in range(len(wl.n_elems)):
            # (past the first NaN only the other rods, which must not see it)
            if r == 2 and steps == 30 and precision == FP64:
                continue
            for tag in STATE:
                a, b = wave.get_rod(tag, r), ref.get_rod(tag, r)
                assert np.isfinite(a).all() and np.array_equal(a, b), (steps, r, tag)
