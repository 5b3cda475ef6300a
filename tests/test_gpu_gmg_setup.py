"""Gmg(...) makes the levels; what only solve and twoVcycle use (stencil
bits, launch programs) is made by the first solve or the second twoVcycle.
And hierarchies of larger grids against the oracle, bit for bit."""
import os
import subprocess
import sys

import numpy as np
import pytest

import fluid2d_amd as F
from fluid2d_amd.device import DeviceArray
from oracle import oracle as orc
from tests.test_gpu_gmg import corner_mask

pytestmark = pytest.mark.gpu
REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# free device memory, from the HIP runtime that the library uses; in a process
# of its own, since that runtime keeps some of what earlier tests gave back
FREE = """
import ctypes as C, gc
import numpy as np
import fluid2d_amd as F
from fluid2d_amd.device import DeviceArray

def free():
    f, t = C.c_size_t(), C.c_size_t()
    assert F.load().f2d_synchronize() == 0
    assert F.load().hipMemGetInfo(C.byref(f), C.byref(t)) == 0
    return f.value
"""


def child(code):
    """What the code prints, as integers."""
    r = subprocess.run([sys.executable, "-c", FREE + code], cwd=REPO, timeout=60,
                       stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    return [int(v) for v in r.stdout.split()]


@pytest.mark.parametrize("first", ["solve", "twoVcycle"])
def test_fused_cycles_are_made_by_the_first_solve(first):
    n = 2048
    made, again, one, two = child("""
n = %d
msk = np.zeros((n + 6, n + 6), np.int8)
msk[3:-3, 3:-3] = 1
x, b = DeviceArray.zeros(msk.shape), DeviceArray.from_host(msk.astype(np.float64))
gm = F.Gmg(dict(n=n, m=n, nh=3, dx=1.0 / n, dy=1.0 / n), msk)
for k in range(50):  # the set-up's own arrays are given back by and by
    gm.Vcycle(0)
    free()
print(free())
gm.Vcycle(0)
print(free())
for k in range(2):
    gm.%s(x, b)
    print(free())
""" % (n, first))
    bits = (n + 6) ** 2  # a byte of stencil bits per cell; the programs come on top
    assert made - again < bits
    if first == "twoVcycle":
        assert made - one < bits  # not worth it for one
    assert made - two >= bits


@pytest.mark.parametrize("nx,ny,geom", [(1024, 768, "xchannel"), (1536, 512, "closed")])
def test_large_hierarchy_vs_oracle(nx, ny, geom):
    g = F.Grid(F.Param(nx=nx, ny=ny, Lx=nx / ny, Ly=1.0, geometry=geom))
    mskp = corner_mask(g)
    gm = F.Gmg(dict(n=nx, m=ny, nh=3, dx=g.dx, dy=g.dy), mskp)
    og = orc.OracleGmg(nx, ny, g.dx, g.dy, mskp)
    b = np.random.default_rng(nx).standard_normal(mskp.shape) * mskp
    g.fill_halo(b)
    xo, xd, bd = np.zeros(b.shape), DeviceArray.zeros(b.shape), DeviceArray.from_host(b)
    for turn in range(2):
        assert gm.solve(xd, bd)[0] == og.solve(xo, b)[0]
        gm.twoVcycle(xd, bd)
        og.twoVcycle(xo, b)
        assert np.array_equal(xd.get(), xo), turn
