"""Kernel-level reductions from several host threads at once: each thread's
result is in its own pinned values, so it equals the one a single thread gets
bit for bit; threads that end hand their values to later ones."""
import threading

import numpy as np
import pytest

from fluid2d_amd import kernels as K
from fluid2d_amd.device import DeviceArray

pytestmark = pytest.mark.gpu
NH = 3


def test_reductions_from_threads():
    rng = np.random.default_rng(2)
    msk = DeviceArray.from_host(np.ones((70, 102), np.int8))
    f = [DeviceArray.from_host((k + 1) * rng.standard_normal((70, 102))) for k in range(6)]

    def call(x):
        return (K.computenorm(msk, x, NH), K.computesumandnorm(msk, x, NH),
                K.computekemaxu(msk, x, x, NH), K.domain_integration(x))
    want = [call(x) for x in f]
    assert len(set(want)) == len(f)
    for turn in range(3):
        got = [set() for _ in f]
        errors = []

        def work(k):
            try:
                for _ in range(50):
                    got[k].add(call(f[k]))
            except Exception as e:
                errors.append(e)
        ts = [threading.Thread(target=work, args=(k,)) for k in range(len(f))]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
        assert not errors
        assert got == [{w} for w in want], turn
