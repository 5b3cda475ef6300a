"""The autotuner times a launch configuration once: the coarse kernel's
one-wavefront threshold is tried only on batches that launch the generic
coarse kernel, which alone knows it."""
import pytest

from fluid2d_amd import autotune
from tests.test_gpu_engine import spec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,Lx,generic", [(64, 64, 1.0, False), (128, 16, 8.0, True)])
def test_one_trial_per_configuration(nx, ny, Lx, generic):
    s = [spec("euler", nx, ny, Lx, 1.0, "closed")]
    cands = [{"coarse_lds_budget": 0, "min_tiles": mt, "coarse_wave_cells": wc}
             for mt in (0, 4096) for wc in (256, 0)]
    best, table = autotune.tune(s, "fp64", steps=1, cands=cands, use_cache=False)
    assert [c["min_tiles"] for c, _ in table] == ([0, 0, 4096, 4096] if generic else [0, 4096])
    assert best in [c for c, _ in table]
    b = autotune.Batch(autotune._pg(s), precision="fp64", tuning=best)
    assert (b.coarse_generic() > 0) == generic
