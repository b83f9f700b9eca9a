"""Fused colour pairs at the finest level on grids whose rows do not fill a workgroup (idle threads, a partial
last workgroup, workgroups past the last row) and on those whose rows are whole in a wave (neighbours exchanged
between lanes), against the FP64 oracle with the tolerance of the FP32 sweep tests."""
import numpy as np
import pytest

import homo3d_amd

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a.astype(np.float64) - b) / np.linalg.norm(b)


@pytest.mark.parametrize("n", [16, 20, 28, 32, 40, 48, 56, 64])
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


@pytest.mark.parametrize("n", [16, 28, 32, 64])
def test_residual(orc, n):
    print("residual: n=%d" % n, flush=True)
    hom = homo3d_amd.Homogenization(homo3d_amd.HomoConfig(reso=n, solver="mg", coarse_half=False))
    x = (homo3d_amd.randc_density(n, 9, 0.3, "none").astype(np.float64) ** 3).astype(np.float32)
    hom.update(x)
    mg = orc.MG(n, 10.0, 0.3)
    mg.set_density(x.astype(np.float64))
    rng = np.random.default_rng(n)
    u = (rng.standard_normal(hom.level_shape(0)) * 0.1).astype(np.float32)
    u[:, :, 0] = 0
    f = rng.standard_normal(hom.level_shape(0)).astype(np.float32)
    hom.set_field(0, 0, u)
    hom.set_field(0, 1, f)
    hom.residual(0)
    got = hom.get_field(0, 2)
    for s in (0, 3, 5):
        # 81 FP32 products a row, as the parity tests' residuals
        assert rel(got[s], orc.residual(n, mg.KE, mg.w, u[s].astype(np.float64), f[s].astype(np.float64))) < 2e-6, s
