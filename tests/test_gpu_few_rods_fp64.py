"""Few FP64 rods of 257 to 512 elements beside shorter ones: all of them are
pieces of one group of tiles, the shorter ones whole, and bitwise what they are
in tiles that hold every rod, with clamps, forces and budgets on either kind."""
import numpy as np
import pytest

from elasticapp_amd import FP64, RAMP_LINEAR
from elasticapp_amd.workloads import build_block
from tests.gpu_helpers import STATE, random_workload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("halo", [0, 6, 31])
@pytest.mark.parametrize("lengths", [[300, 2, 40, 256], [257, 3, 512], [400] + [2] * 130 + [7]])
def test_whole_rods_beside_pieces(lengths, halo):
    wl = random_workload(0, 0, 0, seed=1200 + len(lengths), lengths=lengths)
    last = len(lengths) - 1
    for r in (0, 1, last):
        for i in (0, lengths[r]):
            st = wl.states[r]
            wl.clamps.append((r, st["Position"][:, i].copy(), st["Director"][:, min(i, lengths[r] - 1)].copy(), i))
    wl.forces[last] = (last, wl.forces[last][1], RAMP_LINEAR, 0.0, 30 * wl.dt)
    cut, whole = build_block(wl), build_block(wl)
    cut.set_fused_pieces(0, 0, halo)
    whole.set_fused_config(1024, 2, 0)
    for k, n in enumerate((16, 133, 20)):
        for blk in (cut, whole):
            if k == 1:
                blk.set_step_budget(0, 77)
                blk.set_step_budget(last, 20)
            blk.step_fused(n, FP64)
        assert cut.fused_pieces()[0] == 256 or halo > n or k  # (the plan ends when the first budget in it does)
        for r in range(len(lengths)):
            for tag in STATE:
                assert np.array_equal(whole.get_rod(tag, r), cut.get_rod(tag, r)), (k, r, tag)
        assert np.array_equal(whole.rod_time(), cut.rod_time())
