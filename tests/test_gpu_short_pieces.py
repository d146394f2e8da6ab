"""Pieces whose halo is longer than the part they own: their halos reach past
the neighbouring pieces and end where the rod ends, which several pieces then
hold.  Bitwise the rods stepped whole, hooks at both ends, clocks and budgets
included."""
import numpy as np
import pytest

from elasticapp_amd import FP32_BULK, FP64, RAMP_LINEAR
from elasticapp_amd.workloads import build_block
from tests.gpu_helpers import STATE, random_workload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [FP64, FP32_BULK])
@pytest.mark.parametrize("lanes,epl,halo", [(64, 1, 20), (64, 1, 24), (64, 1, 31), (128, 1, 48), (128, 2, 60), (512, 2, 250)])
def test_halos_longer_than_the_parts(lanes, epl, halo, precision):
    run = halo // 2
    wl = random_workload(0, 0, 0, seed=900 + halo, lengths=[lanes + 1, lanes + 9, 3 * lanes // 2 - 1, min(1000, 3 * lanes)])
    for r in (0, 2):
        n = wl.n_elems[r]
        for i in (0, n):
            st = wl.states[r]
            wl.clamps.append((r, st["Position"][:, i].copy(), st["Director"][:, min(i, n - 1)].copy(), i))
    wl.forces[1] = (1, wl.forces[1][1], RAMP_LINEAR, 0.0, 9 * wl.dt)
    whole, cut = build_block(wl), build_block(wl)
    whole.set_fused_config(1024, 2, run)
    cut.set_fused_config(1024, 2, 4 * run)  # (launches that end where runs do)
    cut.set_fused_pieces(lanes, epl, halo)
    for blk in (whole, cut):
        blk.set_step_budget(3, run + 2)
        for n in (1, halo, 3 * halo + 1):
            blk.step_fused(n, precision)
    for r in range(len(wl.n_elems)):
        for tag in STATE:
            assert np.array_equal(whole.get_rod(tag, r), cut.get_rod(tag, r)), (r, tag)
    assert np.array_equal(whole.rod_time(), cut.rod_time())
