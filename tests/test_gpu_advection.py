"""The kernel-level advection on wavefronts whose cells have the full fluid
window and on those at walls and islands (150 x 40, three 64-column
workgroups a row, the last one clipped), against the oracle: the same bits.
The log-cosh splitting calls the device's log and cosh: a few units in the
last place of the splitting speed, so 1e-13 of the largest flux."""
import numpy as np
import pytest

from fluid2d_amd import kernels as K
from oracle import oracle as orc
from tests.test_gpu_kernels import D, NH, same

pytestmark = pytest.mark.gpu


def fields(walls):
    rng = np.random.default_rng(11)
    m, n = 40 + 2 * NH, 150 + 2 * NH
    msk = np.ones((m, n), np.int8)
    if walls:
        msk[:NH], msk[-NH:], msk[:, :NH], msk[:, -NH:] = 0, 0, 0, 0
        msk[20:24, 30:33] = 0
        msk[10, 140] = 0
    x, u, v = (rng.standard_normal((m, n)) for _ in range(3))
    umax = float((np.abs(u) + np.abs(v)).max())
    return msk, x, u, v, [0.01, 0.02, 2.0, umax, 0.05]


@pytest.mark.parametrize("walls", [False, True])
def test_advection_vs_oracle(walls):
    msk, x, u, v, cst = fields(walls)
    dm, dx, du, dv = D(msk), D(x), D(u), D(v)
    for method in (0, 1, 2):
        for order in (1, 3, 5):
            y, ref = D(np.zeros_like(x)), np.zeros_like(x)
            print("case", walls, method, order, flush=True)
            K.adv_upwind(dm, dx, y, du, dv, cst, NH, method, order)
            orc.adv_upwind(msk, x, ref, u, v, cst, NH, method, order)
            if method < 2:
                same(y.get(), ref, "upwind %d %d" % (method, order))
            else:
                big = cst[3] * np.abs(x).max() * (1 / cst[0] + 1 / cst[1])
                assert np.abs(y.get() - ref).max() <= 1e-13 * big
    for order in (2, 4, 6):
        y, ref = D(np.zeros_like(x)), np.zeros_like(x)
        K.adv_centered(dm, dx, y, du, dv, cst, NH, 0, order)
        orc.adv_centered(msk, x, ref, u, v, cst, NH, order)
        same(y.get(), ref, "centred %d" % order)
