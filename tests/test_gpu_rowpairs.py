"""Fused colour pairs at the finest level on grids whose rows do not fill a workgroup (idle threads, a partial
last workgroup, workgroups past the last row), against the FP64 oracle with the tolerance of the FP32 sweep
tests."""
import numpy as np
import pytest

import homo3d_amd

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a.astype(np.float64) - b) / np.linalg.norm(b)


@pytest.mark.parametrize("n", [20, 28, 40, 48, 56])
@pytest.mark.parametrize("reverse", [False, True])
def test_sweep(orc, n, reverse):
    print("sweep: n=%d reverse=%d" % (n, reverse), flush=True)
    hom = homo3d_amd.Homogenization(homo3d_amd.HomoConfig(reso=n, solver="mg", coarse_half=False))
    x = (homo3d_amd.randc_density(n, 7, 0.3, "none").astype(np.float64) ** 3).astype(np.float32)
    hom.update(x)
    mg = orc.MG(n, 10.0, 0.3)
    mg.set_density(x.astype(np.float64))
    rng = np.random.default_rng(n)
    u = (rng.standard_normal(hom.level_shape(0)) * 0.1).astype(np.float32)
    f = rng.standard_normal(hom.level_shape(0)).astype(np.float32)
    hom.set_field(0, 0, u)
    hom.set_field(0, 1, f)
    hom.smooth(0, 1.0, reverse)
    got = hom.get_field(0, 0)
    for s in (0, 3, 5):
        ref = orc.gs_fine(n, mg.KE, mg.w, u[s].astype(np.float64), f[s].astype(np.float64), 1.0, reverse)
        assert rel(got[s], ref) < 2e-5, s
