"""Patches of a body in compression."""
import time

import pytest

import pymfc

pytestmark = pytest.mark.gpu


def test_compression_keeps_the_patches_copy():
    """Behind the impact's shock the density is up to 6 % higher and a window holds up to 538 candidates
    where the lattice has 504: the patches are planned to hold them. The steps there take 1.25 times
    as long as those before the contact (as many pairs more, and returns); with some patches read
    from memory it was twice as long."""
    s = pymfc.Sim(pymfc.config_impact(200, pymfc.PREC_FP32C, adaptive=False))
    s.step(16)
    times = []
    for _ in range(4):
        s.sync()
        t = time.perf_counter()
        s.step(100)
        s.sync()
        times.append(time.perf_counter() - t)
    assert max(times[2:]) < 1.6 * times[0], times
