"""Smoother tiles of 16 and 8 rows on grids that neither the rows nor the 64
columns divide, against the oracle at the FP64 bar (rel-L2 <= 1e-12 per
field): clipped tiles, wall tiles (masked prolongation) and fluid ones, the
finest level's stencil bits and the explicit operator below it."""
import pytest

from fluid2d_amd.batch import Batch
from tests.test_gpu_engine import TOL, dt_for, init_fields, oracle_for, rel, spec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("min_tiles", [1, 16, 100])
@pytest.mark.parametrize("kind,nx,ny,Lx,Ly,geom", [
    ("euler", 96, 96, 1.0, 1.0, "closed"),
    ("euler", 160, 96, 1.0, 0.6, "perio"),
    ("euler", 192, 192, 1.0, 1.0, "disc"),
    ("boussinesq", 384, 192, 2.0, 1.0, "xchannel"),
])
def test_tile_heights_vs_oracle(kind, nx, ny, Lx, Ly, geom, min_tiles):
    kw = dict(diffusion=True, Kdiff=1e-5) if kind == "boussinesq" else {}
    b = Batch([spec(kind, nx, ny, Lx, Ly, geom, **kw)],
              tuning={"min_tiles": min_tiles, "coarse_lds_budget": 0, "coarse_wave_cells": 0})
    f = init_fields(b, 0, 7)
    b.set_psi_from_vorticity()
    o = oracle_for(b, 0, f)
    dt = dt_for(b, 0, b.diagnostics(0)["maxspeed"])
    b.set_dt(dt)
    b.step(4)
    o.run(4, dt)
    s = b.state(0)
    for k in range(s.shape[0]):
        assert rel(s[k], o.state[k]) <= TOL, (geom, nx, ny, min_tiles, k)
