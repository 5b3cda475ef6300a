"""The coarse kernel's level slots (f2d_coarse.h): grids whose coarse levels
start in every slot and end at every coarsest shape (4 x 4 by lane moves, the
others through LDS; interiors narrower than two halos), and one whose
coarsest level exceeds a wavefront (the generic kernel).  FP64 is the
reference's arithmetic operation for operation, so the state equals the
oracle's bit for bit."""
import numpy as np
import pytest

from fluid2d_amd.batch import Batch
from tests.test_gpu_engine import oracle_for, spec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,geom", [
    (8, 8, "closed"),       # coarsest level alone (slot 4)
    (12, 12, "perio"),      # 6 x 6 over 3 x 3
    (16, 16, "closed"),     # 8 x 8 over 4 x 4
    (32, 16, "xchannel"),   # 16 x 8 over 8 x 4
    (64, 16, "closed"),     # 32 x 8 over 16 x 4
    (32, 64, "closed"),     # taller than wide
    (24, 24, "perio"),      # 12 x 12, 6 x 6, 3 x 3
    (48, 24, "disc"),       # strips of 4 rows on 12 rows
    (80, 48, "closed"),     # 40 x 24, coarsest 5 x 3
    (64, 64, "disc"),       # 1024 cells
    (96, 48, "closed"),     # strips of 8 rows
    (128, 16, "closed"),    # coarsest 32 x 4: the generic kernel
])
def test_coarse_levels_vs_oracle(nx, ny, geom):
    b = Batch([spec("euler", nx, ny, nx / ny, 1.0, geom)])
    g = b.grids[0]
    w = np.random.default_rng(9).standard_normal(g.msk.shape) * g.msk
    g.fill_halo(w)
    b.set_field(0, "vorticity", w)
    b.set_psi_from_vorticity()
    o = oracle_for(b, 0, {"vorticity": w})
    print("case coarse", nx, ny, geom, b.info(0), flush=True)
    dt = 0.8 * min(g.dx, g.dy) / b.diagnostics(0)["maxspeed"]
    b.set_dt(dt)
    b.step(3)
    o.run(3, dt)
    s = b.state(0)
    for k in range(s.shape[0]):
        assert np.array_equal(s[k], o.state[k]), "field %d" % k
