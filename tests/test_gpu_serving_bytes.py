"""The estimate of a pool's device memory, which admission to the serving
loop's budget relies on, holds for every class of grid: it is at least what
creating the pool and stepping it takes, but for the allocator's rounding of
each of a batch's ten arrays to 2 MiB."""
import pytest

from tests.test_gpu_gmg_setup import child

pytestmark = pytest.mark.gpu
ROUNDING = 10 * (2 << 20)


@pytest.mark.parametrize("precision", ["mixed", "fp64"])
@pytest.mark.parametrize("model,n,slots", [
    ("euler", 64, 96), ("euler", 128, 96), ("boussinesq", 128, 64), ("euler", 256, 16),
    ("boussinesq", 256, 4), ("euler", 512, 1), ("euler", 512, 4), ("boussinesq", 1024, 2),
])
def test_pool_estimate_covers_the_pool(precision, model, n, slots):
    used, estimate = child("""
from fluid2d_amd.serving import Pool
Pool((%r, 64), 1, %r).batch.step(1)  # modules and streams
gc.collect()
before = free()
p = Pool((%r, %d), %d, %r)
p.batch.set_psi_from_vorticity()
p.batch.set_steps(1)
p.batch.step(1)
print(before - free(), p.bytes)
""" % (model, precision, model, n, slots, precision))
    print("case pool bytes", precision, model, n, slots, used, estimate, flush=True)
    assert used <= estimate + ROUNDING
    # and not a multiple of it (the smallest grids: mostly lists)
    assert estimate <= 1.35 * used + slots * (1 << 20)
