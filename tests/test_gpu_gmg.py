"""Gmg.solve and Gmg.twoVcycle on the engine's fused kernels against the
oracle, bit for bit (FP64, the reference's operations in its order): grids
the tiles do not divide, a 5-point operator (dx != dy), disc masks, the
Helmholtz shift, a coarsest level beyond a wavefront, and one-level grids,
which keep one launch per routine; calls interleaved with the level-wise
cycles, which share the level arrays."""
import numpy as np
import pytest

import fluid2d_amd as F
from fluid2d_amd.device import DeviceArray
from oracle import oracle as orc

pytestmark = pytest.mark.gpu
NH = 3


def corner_mask(g):
    m = np.zeros_like(g.msk)
    m[:-1, :-1] = (g.msk[:-1, :-1] + g.msk[:-1, 1:] + g.msk[1:, :-1] + g.msk[1:, 1:]) == 4
    return m


@pytest.mark.parametrize("nx,ny,Lx,geom,Rd", [
    (4, 4, 1.0, "perio", None),
    (8, 8, 1.0, "closed", None),
    (48, 96, 0.5, "closed", None),
    (160, 96, 1.0, "perio", None),
    (128, 16, 8.0, "xchannel", None),
    (192, 128, 1.5, "disc", None),
    (512, 256, 2.0, "closed", 0.1),
    (384, 384, 1.3, "xchannel", None),
])
def test_solve_and_two_vcycles_vs_oracle(nx, ny, Lx, geom, Rd):
    g = F.Grid(F.Param(nx=nx, ny=ny, Lx=Lx, Ly=1.0, geometry=geom))
    mskp = corner_mask(g)
    prm = dict(n=nx, m=ny, nh=NH, dx=g.dx, dy=g.dy)
    if Rd:
        prm.update(qgoperator=True, Rd=Rd)
    print("case gmg", nx, ny, Lx, geom, Rd, flush=True)
    gm = F.Gmg(prm, mskp)
    og = orc.OracleGmg(nx, ny, g.dx, g.dy, mskp, Rd=Rd)
    rng = np.random.default_rng(nx + ny)
    for turn in range(2):  # replayed graphs, arrays left by the turn before
        b = rng.standard_normal(mskp.shape) * mskp
        g.fill_halo(b)
        x = rng.standard_normal(mskp.shape) * mskp
        g.fill_halo(x)
        xd, xo, bd = DeviceArray.from_host(x), x.copy(), DeviceArray.from_host(b)
        gm.twoVcycle(xd, bd)
        og.twoVcycle(xo, b)
        assert np.array_equal(xd.get(), xo), ("twoVcycle", turn)
        gm.level(0, "x").upload(x)
        gm.level(0, "b").upload(b)
        og.x(0)[...], og.b(0)[...] = x, b
        gm.Vcycle(0)
        og.Vcycle(0)
        assert np.array_equal(gm.level(0, "x").get(), og.x(0)), ("Vcycle", turn)
        xd.upload(x)
        xo = x.copy()
        nite, _ = gm.solve(xd, bd)
        onite = og.solve(xo, b)[0]
        assert nite == onite
        assert np.array_equal(xd.get(), xo), ("solve", turn)
