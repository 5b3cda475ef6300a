"""The reductions over sizes at the edges of their splits: the NumPy-order
sum (chunks of 8192, halvings that are not equal, leaves of fewer than 8
values, rows a group of eight straddles) equals numpy.sum bit for bit; the
masked sums, which add in a tree, lie within 2^-53 times the depth of the
longest chain (at most 32 columns by rows per thread plus two trees, below
200) of the sum of the terms' magnitudes; the maximum is exact."""
import numpy as np
import pytest

from fluid2d_amd import kernels as K
from fluid2d_amd.device import DeviceArray
from oracle import oracle as orc

pytestmark = pytest.mark.gpu
NH = 3
D = DeviceArray.from_host


@pytest.mark.parametrize("ny,nx", [
    (3, 3), (5, 7), (4, 32), (11, 13), (3, 515), (37, 111), (91, 90), (91, 91), (127, 129),
    (64, 96), (4100, 5), (6, 4099), (1025, 513),
])
def test_sums_at_split_edges(ny, nx):
    rng = np.random.default_rng(ny * 10007 + nx)
    print("case sums", ny, nx, flush=True)
    x, y, u, v = (rng.standard_normal((ny + 2 * NH, nx + 2 * NH)) for _ in range(4))
    msk = (rng.random(x.shape) < 0.8).astype(np.int8)
    inner = (slice(NH, -NH), slice(NH, -NH))
    assert K.domain_integration(D(x)) == np.sum(x[inner])
    f = msk[inner] == 1
    eps = 200 * 2.0 ** -53

    def near(got, terms):
        assert abs(got - np.sum(terms, dtype=np.longdouble)) <= eps * np.abs(terms).sum()
    near(K.computenorm(D(msk), D(x), NH), x[inner][f] ** 2)
    near(K.computedotprod(D(msk), D(x), D(y), NH), (x * y)[inner][f])
    near(K.computesum(D(msk), D(x), NH), x[inner][f])
    s, s2 = K.computesumandnorm(D(msk), D(x), NH)
    near(s, x[inner][f])
    near(s2, x[inner][f] ** 2)
    ke, mx = K.computekemaxu(D(msk), D(u), D(v), NH)
    oke, omx = orc.kemaxu(msk, u, v, NH)
    assert mx == omx
    assert abs(ke - oke) <= (eps + ny * nx * 2.0 ** -53) * abs(oke)  # the oracle adds serially
