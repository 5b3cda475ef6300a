"""Thin grids, whose coarsest level (256 x 4 cells under 1024 x 16) is larger
than the fused coarse kernels take: the hierarchy and the operator-level
model exist and equal the oracle bit for bit, as on every other grid."""
import numpy as np
import pytest

import fluid2d_amd as F
from fluid2d_amd import workloads
from fluid2d_amd.device import DeviceArray
from oracle import oracle as orc
from tests.test_gpu_gmg import corner_mask

pytestmark = pytest.mark.gpu
NH = 3


@pytest.mark.parametrize("nx,ny,Lx,geom,Rd", [
    (1024, 16, 64.0, "xchannel", None),
    (16, 1024, 0.02, "closed", None),
    (8, 480, 1.0, "perio", 0.1),
])
def test_thin_hierarchy_vs_oracle(nx, ny, Lx, geom, Rd):
    g = F.Grid(F.Param(nx=nx, ny=ny, Lx=Lx, Ly=1.0, geometry=geom))
    mskp = corner_mask(g)
    prm = dict(n=nx, m=ny, nh=NH, dx=g.dx, dy=g.dy)
    if Rd:
        prm.update(qgoperator=True, Rd=Rd)
    print("case thin gmg", nx, ny, Lx, geom, Rd, flush=True)
    gm = F.Gmg(prm, mskp)
    og = orc.OracleGmg(nx, ny, g.dx, g.dy, mskp, Rd=Rd)
    assert gm.nlevs == og.nlevs
    rng = np.random.default_rng(nx + ny)
    b, x = (rng.standard_normal(mskp.shape) * mskp for _ in range(2))
    g.fill_halo(b)
    g.fill_halo(x)
    xd, bd = DeviceArray.from_host(x), DeviceArray.from_host(b)
    for turn in range(2):
        xd.upload(x)
        xo = x.copy()
        gm.twoVcycle(xd, bd)
        og.twoVcycle(xo, b)
        assert np.array_equal(xd.get(), xo), turn
    xd.upload(x)
    xo = x.copy()
    nite, _ = gm.solve(xd, bd)
    assert nite == og.solve(xo, b)[0]
    assert np.array_equal(xd.get(), xo)


def test_thin_model_vs_oracle():
    nx, ny, Lx = 1024, 16, 64.0
    p = F.Param(modelname="euler", nx=nx, ny=ny, Lx=Lx, Ly=1.0, geometry="xchannel", engine=False)
    g = F.Grid(p)
    f = F.Fluid2d(p, g)
    o = orc.OracleModel("euler", nx, ny, Lx, 1.0, geometry="xchannel")
    w = workloads.turbulence(g, 3)
    f.model.var.get("vorticity")[...] = w
    o.get("vorticity")[...] = w
    f.model.set_psi_from_vorticity()
    o.set_psi_from_vorticity()
    # both start from their own maxspeed (core/fluid2d.py:199)
    umax = f.model.diagnostics(f.model.var, 0.)["maxspeed"]
    assert umax == o.diagnostics()["maxspeed"]
    dt = 0.5 * min(g.dx, g.dy) / umax
    f.model.run(2, dt)
    o.run(2, dt)
    s = f.model.var.state
    for k in range(s.shape[0]):
        assert np.array_equal(s[k], o.state[k]), k
