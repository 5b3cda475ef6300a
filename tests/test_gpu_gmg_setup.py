"""Gmg(...) makes the levels; what only solve and twoVcycle use (stencil
bits, launch programs) is made by the first solve or the second twoVcycle."""
import numpy as np
import pytest

import fluid2d_amd as F
from fluid2d_amd.device import DeviceArray

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("first", ["solve", "twoVcycle"])
def test_fused_cycles_are_made_by_the_first_solve(first):
    import torch
    n = 2048
    msk = np.zeros((n + 6, n + 6), np.int8)
    msk[3:-3, 3:-3] = 1
    x, b = DeviceArray.zeros(msk.shape), DeviceArray.from_host(msk.astype(np.float64))
    gm = F.Gmg(dict(n=n, m=n, nh=3, dx=1.0 / n, dy=1.0 / n), msk)

    def free():
        torch.cuda.synchronize()
        return torch.cuda.mem_get_info()[0]
    before = free()
    gm.Vcycle(0)
    if first == "twoVcycle":  # not worth it for one
        gm.twoVcycle(x, b)
    assert free() == before
    getattr(gm, first)(x, b)
    after = free()
    assert before - after >= msk.size  # a byte of stencil bits per cell, and the programs
    gm.solve(x, b)
    gm.solve(x, b)
    assert before - free() <= 2 * (before - after)
