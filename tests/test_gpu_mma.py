"""GPU MMA step at every constraint count the kernels are compiled for, on variable counts around a wave
and a workgroup (1, 64, 257, 300), against the FP64 oracle over the iterations that change the asymptotes.
"""
import numpy as np
import pytest

import homo3d_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m", [(1, 1), (64, 2), (257, 3), (300, 4)])
def test_mma_constraint_counts(orc, n, m):
    print("mma: n=%d m=%d" % (n, m), flush=True)
    rng = np.random.default_rng(100 * n + m)
    x = rng.uniform(0.2, 0.8, n)
    gpu = homo3d_amd.MMAOptimizer(m, n, 1.0, 0.0, 1000.0, 1.0)
    gpu.setBound(0.001, 1.0)
    st = {"x": x.copy(), "xmin": np.full(n, 0.001), "xmax": np.ones(n), "xold1": x.copy(), "xold2": x.copy(),
          "low": np.zeros(n), "upp": np.zeros(n)}
    w = rng.uniform(0.5, 2.0, (m, n))
    for it in range(5):
        xin = st["x"].astype(np.float32).astype(np.float64)
        st["x"][:] = xin
        df0 = (-(1.0 + np.sin(3 * xin))).astype(np.float32)
        g = np.array([(w[i] * xin).sum() / n - 0.4 - 0.1 * i for i in range(m)], dtype=np.float32)
        dg = (w / n).astype(np.float32)
        xg = gpu.update(it, xin.astype(np.float32), df0, g, list(dg))
        orc.mma_update(st, it, df0.astype(np.float64), g.astype(np.float64), dg.astype(np.float64), 1.0,
                       np.zeros(m), np.full(m, 1000.0), np.ones(m), 1.0)
        x64, lo, up, _ = gpu.state()
        # the same Newton steps in FP64 sums of another order: a few hundred roundings of 1e-16, amplified
        # by the system's conditioning (below 1e4 at these sizes)
        assert np.abs(x64 - st["x"]).max() <= 1e-9, it
        assert np.abs(lo - st["low"]).max() <= 1e-12 and np.abs(up - st["upp"]).max() <= 1e-12
        assert np.array_equal(xg, x64.astype(np.float32))
