"""One MMA step from host arrays (whose result takes the place of the step's copy of the design) and from
device arrays: the same design, state and asymptotes, bit for bit, over the iterations that read the designs
of the two before."""
import ctypes

import numpy as np
import pytest

import homo3d_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m", [(1000, 1), (70001, 2)])
def test_host_and_device_arrays(n, m):
    print("mma arrays: n=%d m=%d" % (n, m), flush=True)
    rng = np.random.default_rng(n)
    x = rng.uniform(0.2, 0.8, n).astype(np.float32)
    w = rng.uniform(0.5, 2.0, (m, n))
    host, dev = (homo3d_amd.MMAOptimizer(m, n, 1.0, 0.0, 1000.0, 1.0) for _ in range(2))
    host.setBound(0.001, 1.0)
    dev.setBound(0.001, 1.0)
    xd = homo3d_amd.DeviceBuffer.from_array(x)
    for it in range(1, 6):
        df = (-(1.0 + np.sin(3 * x.astype(np.float64)))).astype(np.float32)
        g = np.array([(w[i] * x).sum() / n - 0.4 - 0.1 * i for i in range(m)], dtype=np.float32)
        dg = (w / n).astype(np.float32)
        dfd = homo3d_amd.DeviceBuffer.from_array(df)
        dgd = [homo3d_amd.DeviceBuffer.from_array(v) for v in dg]
        ptrs = (ctypes.c_void_p * m)(*[v.value for v in dgd])
        rc = homo3d_amd.lib().homo3d_mma_update(dev._h, it, xd.ptr, dfd.ptr, g.ctypes.data_as(ctypes.c_void_p), ptrs, 1)
        assert rc == homo3d_amd.HOMO3D_OK
        xin = x.copy()
        x = host.update(it, xin, df, g, list(dg))
        assert np.array_equal(xd.download(), x), it
        sh, sd = host.state(), dev.state()
        for a, b in zip(sh[:3], sd[:3]):
            assert np.array_equal(a, b), it
        # the asymptotes are about the design that came in, not the one that went out
        assert np.all(sh[1] < xin) and np.all(sh[2] > xin)
