"""The double sweep of the kernel-level smoother, in one pass (from 196608
cells) at the edges of its 64 x 16 tiles and in two below, on a random
operator, mask and halo, against the oracle: the same bits (same operations in
the same order)."""
import numpy as np
import pytest

from fluid2d_amd import kernels as K
from oracle import oracle as orc
from tests.test_gpu_kernels import D, NH, filled

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ny,nx", [(4, 4), (15, 63), (16, 64), (17, 65), (18, 66), (34, 130),
                                   (5, 200), (97, 6), (256, 192), (448, 448),
                                   (449, 449), (447, 511), (466, 450), (4, 50001), (33000, 6)])
def test_double_sweep_at_tile_edges(ny, nx):
    rng = np.random.default_rng(100 * ny + nx)
    m, n = ny + 2 * NH, nx + 2 * NH
    A = rng.standard_normal((5, m, n))
    A[4] = -4. - np.abs(A[4])
    msk = (rng.random((m, n)) < 0.8).astype(np.int8)
    x, b = rng.standard_normal((m, n)), rng.standard_normal((m, n))
    xs, work = D(x), D(rng.standard_normal((m, n)))
    print("case", ny, nx, flush=True)
    K.smoothtwicewitha_fill(D(msk), D(A), xs, D(b), 8.0 / 9.0, work)
    ref = x.copy()
    orc.smoothtwice(msk, A, ref, b, 8.0 / 9.0)
    assert (xs.get() == filled(ref)).all()
