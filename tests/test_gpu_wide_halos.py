"""Pieces of long rods whose shape is left free take wider halos, and launches
of as many steps, while every piece has a compute unit of its own: bitwise the
pieces with the default halo in launches of its own, both precisions, with
budgets that end inside a launch, clamps in a halo and whole rods beside."""
import numpy as np
import pytest

from elasticapp_amd import FP32_BULK, FP64
from elasticapp_amd.workloads import build_block
from tests.gpu_helpers import STATE, random_workload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [FP64, FP32_BULK])
@pytest.mark.parametrize("lengths", [[1025], [1300, 30, 200, 2000], [5000] * 12 + [3, 250], [5000] * 25])
def test_wide_halos(lengths, precision):
    wl = random_workload(0, 0, 0, seed=1000 + len(lengths), lengths=lengths)
    st = wl.states[0]
    wl.clamps.append((0, st["Position"][:, 300].copy(), st["Director"][:, 300].copy(), 300))
    wide, ref = build_block(wl), build_block(wl)
    wide.step_fused(1, precision)
    lanes, epl, halo, tiles, pieces = wide.fused_pieces()
    assert halo == 16 and pieces >= 2
    ref.set_fused_pieces(lanes, epl, 16)  # (requested: the halo stays; no rod between 256 and 1,024, which it would cut)
    ref.step_fused(1, precision)
    # (wider halos make more pieces; 25 rods leave no room for any)
    assert pieces == ref.fused_pieces()[4] if len(lengths) == 25 else pieces > ref.fused_pieces()[4]
    for k, n in enumerate((15, 64, 133)):
        for b in (wide, ref):
            if k == 2:
                b.set_step_budget(0, 77)
                b.set_step_budget(len(lengths) - 1, 20)
            b.step_fused(n, precision)
    for r in range(len(lengths)):
        for tag in STATE:
            assert np.array_equal(wide.get_rod(tag, r), ref.get_rod(tag, r)), (r, tag)
    assert np.array_equal(wide.rod_time(), ref.rod_time())
