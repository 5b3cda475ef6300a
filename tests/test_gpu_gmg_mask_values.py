"""A corner mask with another value than 0 and 1 at single cells: the level-0
operator holds the stencil weights times mask products
(core/gmg/level.py:292), so it is not the stencil with constant weights, and
solve and twoVcycle have to use the operator as it is (against the oracle,
bit for bit)."""
import numpy as np
import pytest

import fluid2d_amd as F
from fluid2d_amd.device import DeviceArray
from oracle import oracle as orc
from tests.test_gpu_gmg import corner_mask

pytestmark = pytest.mark.gpu
NH = 3


@pytest.mark.parametrize("value", [2, -1])
@pytest.mark.parametrize("j,i", [(33, 33), (20, 41)])  # over and beside a coarse point
def test_other_mask_value_vs_oracle(value, j, i):
    nx = ny = 64
    g = F.Grid(F.Param(nx=nx, ny=ny, Lx=1.0, Ly=1.0, geometry="closed"))
    mskp = corner_mask(g)
    mskp[j, i] = value
    print("case mask value", value, j, i, flush=True)
    gm = F.Gmg(dict(n=nx, m=ny, nh=NH, dx=g.dx, dy=g.dy), mskp)
    og = orc.OracleGmg(nx, ny, g.dx, g.dy, mskp)
    rng = np.random.default_rng(5)
    b, x = (rng.standard_normal(mskp.shape) * (mskp != 0) for _ in range(2))
    g.fill_halo(b)
    g.fill_halo(x)
    bd = DeviceArray.from_host(b)
    for turn in range(2):
        xd, xo = DeviceArray.from_host(x), x.copy()
        gm.twoVcycle(xd, bd)
        og.twoVcycle(xo, b)
        assert np.isfinite(xo).all()
        assert np.array_equal(xd.get(), xo), turn
    xd, xo = DeviceArray.from_host(x), x.copy()
    gm.solve(xd, bd)
    og.solve(xo, b)
    assert np.array_equal(xd.get(), xo)
