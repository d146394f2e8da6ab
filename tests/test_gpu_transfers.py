"""Downloads return what was uploaded, bit for bit, at the sizes where their
path changes: the pinned stages (to 256 KB and 1 MB), the ring of chunks (two
threads, from 2 MB four; 1 MB chunks, from 6 MB 2 MB; past its 4 chunks),
whole fields and strided rods.
"""
import threading

import numpy as np
import pytest

from elasticapp_amd import DeviceBlock

pytestmark = pytest.mark.gpu

TAGS = ("Position", "Director", "Mass")  # 3, 9 and 1 lines


def _check(blk, rng, rounds=2):
    for tag in TAGS:
        for _ in range(rounds):  # (again through buffers that are there)
            a = rng.normal(size=blk.get_field(tag).shape)
            blk.set_field(tag, a)
            assert np.array_equal(blk.get_field(tag), a), tag
        for r, s in enumerate(blk.starts):
            n = blk.rod_slots(tag, r)
            assert np.array_equal(blk.get_rod(tag, r), a[:, s:s + n]), (tag, r)


# Position at 24 B a slot: 256 KB at 10,922 slots, 1 MB at 43,690; Director at
# 72 B: 1 MB at 14,563, 2 MB at 29,127, whole chunks and one value more, and rings that wrap
@pytest.mark.parametrize("n", [2, 10921, 10922, 14563, 14564, 29127, 29128, 43690, 58254, 58255, 116508, 116509, 131071, 131072, 300001])
def test_one_rod(n):
    with DeviceBlock([n]) as blk:
        _check(blk, np.random.default_rng(n))


@pytest.mark.parametrize("lengths", [(2, 3, 5), (3640, 3641, 7), (120000, 2, 11000, 10922)])
def test_rods_of_a_block(lengths):
    with DeviceBlock(list(lengths)) as blk:
        _check(blk, np.random.default_rng(sum(lengths)))


def test_blocks_in_threads():
    """Two host threads, each with its own block."""
    bad = []

    def work(seed):
        try:
            with DeviceBlock([200000, 50]) as blk:
                _check(blk, np.random.default_rng(seed), rounds=3)
        except BaseException as e:  # noqa: B902
            bad.append(e)

    ts = [threading.Thread(target=work, args=(s,)) for s in (1, 2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad, bad
