"""Level arrays handed out by Gmg.level are the hierarchy's own: solve and
twoVcycle work on the operator and mask they hold at the call, as Vcycle
does, bit for bit, and leave the levels' intermediate values where a view
that was handed out before shows them."""
import numpy as np
import pytest

import fluid2d_amd as F
from fluid2d_amd.device import DeviceArray
from tests.test_gpu_gmg import corner_mask

pytestmark = pytest.mark.gpu
NH = 3


def pair(nx, ny):
    """Two equal hierarchies, a mask and fields."""
    g = F.Grid(F.Param(nx=nx, ny=ny, Lx=nx / ny, Ly=1.0, geometry="closed"))
    mskp = corner_mask(g)
    prm = dict(n=nx, m=ny, nh=NH, dx=g.dx, dy=g.dy)
    rng = np.random.default_rng(nx)
    b, x = (rng.standard_normal(mskp.shape) * mskp for _ in range(2))
    g.fill_halo(b)
    g.fill_halo(x)
    return g, prm, mskp, x, b


def by_levels(gm, x, b):
    """twoVcycle by the level-wise cycles."""
    gm.level(0, "x").upload(x)
    gm.level(0, "b").upload(b)
    gm.Vcycle(0)
    gm.Vcycle(0)
    return gm.level(0, "x").get()


@pytest.mark.parametrize("lev", [0, 1, 3])
@pytest.mark.parametrize("used", [False, True])
def test_edited_operator(lev, used):
    g, prm, mskp, x, b = pair(128, 64)
    print("case edited operator", lev, used, flush=True)
    gm, ref = F.Gmg(prm, mskp), F.Gmg(prm, mskp)
    xd, bd = DeviceArray.from_host(x), DeviceArray.from_host(b)
    if used:
        gm.twoVcycle(xd, bd)
        gm.solve(xd, bd)
        xd.upload(x)
    for h in (gm, ref):
        A = h.level(lev, "A")
        a = A.get()
        a[4] *= 1.25  # a stronger centre on every cell
        A.upload(a)
    want = by_levels(ref, x, b)
    for turn in range(2):
        xd.upload(x)
        gm.twoVcycle(xd, bd)
        assert np.array_equal(xd.get(), want), turn


def test_edited_mask():
    g, prm, mskp, x, b = pair(128, 64)
    gm, ref = F.Gmg(prm, mskp), F.Gmg(prm, mskp)
    xd, bd = DeviceArray.from_host(x), DeviceArray.from_host(b)
    for h in (gm, ref):
        M = h.level(2, "msk")
        m = M.get()
        m[8:12, 10:14] = 0
        M.upload(m)
    want = by_levels(ref, x, b)
    for turn in range(2):
        xd.upload(x)
        gm.twoVcycle(xd, bd)
        assert np.array_equal(xd.get(), want), turn


def test_views_show_the_levels():
    g, prm, mskp, x, b = pair(128, 64)
    gm, ref = F.Gmg(prm, mskp), F.Gmg(prm, mskp)
    v = [(lev, w, gm.level(lev, w)) for lev in range(1, gm.nlevs) for w in "xb"]
    v.append((0, "r", gm.level(0, "r")))
    xd, bd = DeviceArray.from_host(x), DeviceArray.from_host(b)
    by_levels(ref, x, b)
    for turn in range(2):
        xd.upload(x)
        gm.twoVcycle(xd, bd)
        for lev, w, a in v:
            assert np.array_equal(a.get(), ref.level(lev, w).get()), (lev, w, turn)
