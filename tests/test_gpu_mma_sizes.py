"""GPU MMA step on variable counts that fill the reductions of its control kernels partly (50001: 196
workgroups), and that exceed one pass of the grid, give the line search fewer workgroups than the other passes
and end in a partial one (300001), against the FP64 oracle."""
import numpy as np
import pytest

import homo3d_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m", [(50001, 2), (50001, 4), (300001, 2)])
def test_mma_large(orc, n, m):
    print("mma: n=%d m=%d" % (n, m), flush=True)
    rng = np.random.default_rng(n)
    x = rng.uniform(0.2, 0.8, n)
    gpu = homo3d_amd.MMAOptimizer(m, n, 1.0, 0.0, 1000.0, 1.0)
    gpu.setBound(0.001, 1.0)
    st = {"x": x.copy(), "xmin": np.full(n, 0.001), "xmax": np.ones(n), "xold1": x.copy(), "xold2": x.copy(),
          "low": np.zeros(n), "upp": np.zeros(n)}
    w = rng.uniform(0.5, 2.0, (m, n))
    for it in range(4):
        xin = st["x"].astype(np.float32).astype(np.float64)
        st["x"][:] = xin
        df0 = (-(1.0 + np.sin(3 * xin))).astype(np.float32)
        g = np.array([1000 * ((w[i] * xin).sum() / n - 0.4 - 0.1 * i) for i in range(m)], dtype=np.float32)
        dg = (1000 * w / n).astype(np.float32)
        xg = gpu.update(it, xin.astype(np.float32), df0, g, list(dg))
        orc.mma_update(st, it, df0.astype(np.float64), g.astype(np.float64), dg.astype(np.float64), 1.0,
                       np.zeros(m), np.full(m, 1000.0), np.ones(m), 1.0)
        x64, lo, up, _ = gpu.state()
        # sums of another order: reordering the oracle's own moves its x by 5e-14 at these sizes; the other
        # MMA tests allow as much
        assert np.abs(x64 - st["x"]).max() <= 1e-9, it
        assert np.abs(lo - st["low"]).max() <= 1e-12 and np.abs(up - st["upp"]).max() <= 1e-12
        assert np.array_equal(xg, x64.astype(np.float32))
