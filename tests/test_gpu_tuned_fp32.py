"""An autotuned FP32-bulk batch of rods of up to 512 elements returns what an
untuned one does, bit for bit: the trials leave the rods whole."""
import numpy as np
import pytest

from elasticapp_amd import FP32_BULK
from elasticapp_amd.workloads import build_block
from tests.gpu_helpers import STATE, random_workload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lengths", [[105, 258, 130, 200, 150, 180], [25, 314, 60, 100], [3, 512], [92, 132] * 200])
def test_tuned_fp32_equals_untuned(lengths):
    wl = random_workload(0, 0, 0, seed=1300 + lengths[0], lengths=lengths)
    tuned, free = build_block(wl), build_block(wl)
    tuned.autotune(FP32_BULK, 50)
    for n in (100, 7, 230):
        for blk in (tuned, free):
            blk.step_fused(n, FP32_BULK)
    for tag in STATE:
        for r in range(len(lengths)):
            assert np.array_equal(tuned.get_rod(tag, r), free.get_rod(tag, r)), (tag, r)
    assert np.array_equal(tuned.rod_time(), free.rod_time())
