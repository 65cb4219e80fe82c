"""Sizes of the groups that fits launched together get: no more workgroups than
the device holds, whatever the number of host threads (no GPU work)."""
import contextlib
import importlib
import threading

import pytest


@pytest.fixture
def F():
    return importlib.import_module("2018_dictionary_tomography_amd.fit")


def _together(count, angles, room, groups):
    with contextlib.ExitStack() as s:
        return [s.enter_context(count.take("gpu", nA, room, g)) for nA, g in zip(angles, groups)]


@pytest.mark.parametrize("angles,n", [(61, 64), (61, 100), (20, 128), (4, 300), (200, 40), (256, 64)])
def test_never_more_than_the_device_holds(F, angles, n):
    count = F.WorkgroupCount()
    got = _together(count, [angles] * n, 256, [None] * n)
    assert got[0] == F.default_group(angles) and min(got) >= 1
    # a single workgroup waits for nobody, so it may wait for a place
    assert sum(g for g in got if g > 1) <= 256
    # 16 angles per workgroup beside other fits: as many at once as the device holds of those
    share = max(1, min(8, -(-angles // 16)))
    assert sum(g >= share for g in got) >= min(n, 1 + (256 - got[0]) // share)
    # all given back
    assert _together(count, [angles], 256, [None]) == [F.default_group(angles)]


def test_given_groups_and_devices(F):
    count = F.WorkgroupCount()
    assert _together(count, [61] * 3, 256, [200, 200, None]) == [200, 56, 1]
    with count.take("a", 61, 256) as a, count.take("b", 61, 256) as b:
        assert a == b == 8
    with pytest.raises(KeyError):
        with count.take("gpu", 61, 256):
            raise KeyError
    assert _together(count, [61], 4, [None]) == [4]


def test_threads(F):
    count, worst, start = F.WorkgroupCount(), [0], threading.Barrier(16)

    def run():
        start.wait()
        for _ in range(200):
            with count.take("gpu", 128, 64) as g:
                assert g >= 1
                worst[0] = max(worst[0], sum(count._used.values()))

    t = [threading.Thread(target=run) for _ in range(16)]
    for u in t:
        u.start()
    for u in t:
        u.join()
    assert worst[0] <= 64 + 15 and sum(count._used.values()) == 0
