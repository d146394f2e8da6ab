"""The shapes a batch takes when the caller leaves them free: their rule (one
element per thread at 512 lanes while every tile has a CU of its own, and for
FP64; smaller pieces of long rods), calls that alternate between the
precisions on one batch, and results that do not depend on any of it."""
import numpy as np
import pytest

from elasticapp_amd import FP32_BULK, FP64
from elasticapp_amd.workloads import build_block
from tests.gpu_helpers import STATE, random_workload

pytestmark = pytest.mark.gpu


def _same(a, b):
    return all(np.array_equal(a.get_field(t), b.get_field(t)) for t in STATE)


@pytest.mark.parametrize("precision", [FP64, FP32_BULK])
@pytest.mark.parametrize("lengths,config,pieces", [
    ([256, 3], {FP64: (256, 1), FP32_BULK: (256, 1)}, {FP64: 0, FP32_BULK: 0}),
    ([257, 3, 40], {FP64: (256, 1), FP32_BULK: (512, 1)}, {FP64: 256, FP32_BULK: 0}),
    ([512, 2, 511], {FP64: (256, 1), FP32_BULK: (512, 1)}, {FP64: 256, FP32_BULK: 0}),
    ([400] * 400, {FP64: (512, 1), FP32_BULK: (512, 2)}, {FP64: 0, FP32_BULK: 0}),  # more than 256 tiles
    ([513, 20], {FP64: (1024, 2), FP32_BULK: (1024, 2)}, {FP64: 0, FP32_BULK: 0}),
    ([400] * 21 + [20], {FP64: (512, 1), FP32_BULK: (512, 1)}, {FP64: 0, FP32_BULK: 0}),
    ([1025], {FP64: (0, 0), FP32_BULK: (0, 0)}, {FP64: 256, FP32_BULK: 256}),
    ([5000] * 20, {FP64: (0, 0), FP32_BULK: (0, 0)}, {FP64: 512, FP32_BULK: 512}),
    ([5000] * 32 + [700], {FP64: (1024, 2), FP32_BULK: (1024, 2)}, {FP64: 256, FP32_BULK: 1024}),
])
def test_free_shapes(lengths, config, pieces, precision):
    wl = random_workload(0, 0, 0, seed=len(lengths) + lengths[0], lengths=lengths)
    blk, ref = build_block(wl), build_block(wl)
    ref.set_fused_config(1024, 0, 0)  # (a requested shape: its pieces take it too)
    for b in (blk, ref):
        b.step_fused(21, precision)
    assert blk.fused_config()[:2] == config[precision]
    assert blk.fused_pieces()[0] == pieces[precision]
    assert ref.fused_pieces()[0] in (0, 1024)
    assert _same(blk, ref)


@pytest.mark.parametrize("lengths", [[400] * 400, [5000] * 32 + [700], [30, 200]])
def test_alternating_precisions(lengths):
    """FP64 and FP32-bulk calls in turn on one batch, through launches and
    graphs, with rods that run out of steps between them, equal the same calls
    on a batch whose plan is remade before every one."""
    wl = random_workload(0, 0, 0, seed=len(lengths), lengths=lengths)
    a, b = build_block(wl), build_block(wl)
    calls = [(FP64, 5), (FP32_BULK, 6), (FP64, 4), (FP32_BULK, 40), (FP32_BULK, 3), (FP64, 40), (FP64, 7), (FP32_BULK, 40)]
    for k, (precision, n) in enumerate(calls):
        b.set_fused_config(0, 0, 0)  # (invalidates the plan)
        for blk in (a, b):
            if k == 4:
                blk.set_step_budget(0, 20)
            if n == 40:
                blk.step_fused_graph(n, 20, precision)
            else:
                blk.step_fused(n, precision)
        assert _same(a, b), k
        assert np.array_equal(a.rod_time(), b.rod_time()), k
        assert a.fused_config() == b.fused_config() and a.fused_pieces() == b.fused_pieces(), k


@pytest.mark.parametrize("precision", [FP64, FP32_BULK])
@pytest.mark.parametrize("lengths", [[30, 200], [1300, 40]])
def test_a_first_budget_after_a_capture(lengths, precision):
    """A graph captured before any rod had a step budget is captured again once
    one has."""
    wl = random_workload(0, 0, 0, seed=40 + lengths[0], lengths=lengths)
    a, b = build_block(wl), build_block(wl)
    for blk in (a, b):
        blk.set_fused_config(0, 0, 20)
    a.capture_fused_graph(60, precision)
    for n in (60, 120):
        for blk in (a, b):
            if n == 120:
                blk.set_step_budget(0, 50)
        a.step_fused_graph(n, 60, precision)
        b.step_fused(n, precision)
        assert _same(a, b), n
        assert np.array_equal(a.rod_time(), b.rod_time()), n
    assert a.rod_time()[0] < a.rod_time()[1]
