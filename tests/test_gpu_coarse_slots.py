"""The register coarse kernel against the generic one, by level slot, in both
precisions: a batch with one grid outside the slots (128 x 16, coarsest level
32 x 4) runs the generic kernel for all its instances, and the two kernels
apply the same FP64 operations to the same operands, so an instance alone and
in that batch agree bit for bit.  The slot is asserted from the level the
coarse part starts at, so that a case cannot move to another one unseen."""
import numpy as np
import pytest

from fluid2d_amd.batch import Batch
from tests.test_gpu_engine import spec

pytestmark = pytest.mark.gpu
THIN = spec("euler", 128, 16, 8.0, 1.0, "closed")


def run(specs, precision):
    b = Batch(specs, precision=precision)
    for i, g in enumerate(b.grids):
        rng = np.random.default_rng(g.nx + i)
        for name in ("vorticity", "buoyancy")[:1 + (specs[i]["modelname"] == "boussinesq")]:
            a = rng.standard_normal(g.msk.shape) * g.msk
            g.fill_halo(a)
            b.set_field(i, name, a)
    b.set_psi_from_vorticity()
    for i, g in enumerate(b.grids):
        ms = b.diagnostics(i)["maxspeed"]
        b.set_dt(0.5 * min(g.dx, g.dy) / (ms if specs[i]["modelname"] == "euler" else 1.0), i)
    b.step(3)
    return b


@pytest.mark.parametrize("precision,kind,nx,ny,geom,top", [
    ("mixed", "euler", 96, 48, "closed", (24, 48)),       # strips of 8 rows: 24 rows
    ("mixed", "euler", 48, 96, "perio", (48, 24)),        # 48 rows
    ("mixed", "euler", 80, 64, "closed", (32, 40)),       # coarsest 4 x 5
    ("mixed", "euler", 64, 112, "disc", (56, 32)),        # 56 rows, coarsest 7 x 4
    ("mixed", "euler", 48, 128, "closed", (64, 24)),      # all 64 rows
    ("mixed", "boussinesq", 384, 192, "xchannel", (24, 48)),
    ("mixed", "euler", 64, 64, "disc", (32, 32)),         # strips of 4
    ("mixed", "euler", 24, 24, "perio", (12, 12)),        # one cell a thread
    ("mixed", "euler", 16, 16, "closed", (8, 8)),         # one wavefront
    ("mixed", "euler", 8, 8, "closed", (4, 4)),
    ("fp64", "euler", 96, 48, "closed", (12, 24)),        # FP64 never takes 8 rows
    ("fp64", "euler", 64, 64, "disc", (32, 32)),
    ("fp64", "euler", 24, 24, "perio", (12, 12)),
    ("fp64", "euler", 8, 8, "closed", (4, 4)),
])
def test_register_kernel_equals_generic(precision, kind, nx, ny, geom, top):
    s = spec(kind, nx, ny, nx / ny, 1.0, geom)
    print("case coarse slots", precision, kind, nx, ny, geom, flush=True)
    alone = run([s], precision)
    k = alone.info(0)["nfine"]
    assert (ny >> k, nx >> k) == top
    mix = run([s, THIN], precision)
    assert mix.info(0)["nfine"] == k
    assert np.isfinite(alone.state(0)).all()
    assert np.array_equal(alone.state(0), mix.state(0))
    assert alone.solve_info(0)[0] == mix.solve_info(0)[0]
