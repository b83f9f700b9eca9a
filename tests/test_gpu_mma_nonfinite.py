"""MMA steps whose residual norm is not a number: a variable with equal bounds (its asymptotes meet at it), an
infinite entry of a gradient.  The interior point takes no step there, as in the FP64 oracle: the design is the
middle of the move limits, finite, after the same number of Newton steps."""
import numpy as np
import pytest

import homo3d_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["equal bounds", "objective", "constraint"])
@pytest.mark.parametrize("n,m", [(2, 1), (64, 4), (70001, 2)])
def test_no_step_without_a_residual(orc, kind, n, m):
    print("mma: %s n=%d m=%d" % (kind, n, m), flush=True)
    rng = np.random.default_rng(n)
    x = rng.uniform(0.2, 0.8, n).astype(np.float32).astype(np.float64)
    w = rng.uniform(0.5, 2.0, (m, n))
    lo, hi = np.full(n, 0.001, np.float32), np.ones(n, np.float32)
    if kind == "equal bounds":
        lo[0] = hi[0] = x[0]
    gpu = homo3d_amd.MMAOptimizer(m, n, 1.0, 0.0, 1000.0, 1.0)
    gpu.setBound(lo, hi)
    st = {"x": x.copy(), "xmin": lo.astype(np.float64), "xmax": hi.astype(np.float64), "xold1": x.copy(),
          "xold2": x.copy(), "low": np.zeros(n), "upp": np.zeros(n)}
    for it in range(1, 4 if n < 1000 else 2):
        xin = st["x"].astype(np.float32).astype(np.float64)
        st["x"][:] = xin
        df0 = (-(1.0 + np.sin(3 * xin))).astype(np.float32)
        g = np.array([(w[i] * xin).sum() / n - 0.4 - 0.1 * i for i in range(m)], dtype=np.float32)
        dg = (w / n).astype(np.float32)
        if kind == "objective":
            df0[0] = np.inf
        elif kind == "constraint":
            dg[m - 1, n - 1] = -np.inf
        xg = gpu.update(it, xin.astype(np.float32), df0, g, list(dg))
        newton = orc.mma_update(st, it, df0.astype(np.float64), g.astype(np.float64), dg.astype(np.float64), 1.0,
                                np.zeros(m), np.full(m, 1000.0), np.ones(m), 1.0)
        x64, low, upp, steps = gpu.state()
        assert np.isfinite(st["x"]).all() and newton > 0
        assert steps == newton
        assert np.abs(x64 - st["x"]).max() <= 1e-12
        assert np.abs(low - st["low"]).max() <= 1e-12 and np.abs(upp - st["upp"]).max() <= 1e-12
        assert np.array_equal(xg, x64.astype(np.float32))
