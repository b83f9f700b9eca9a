"""Fused colour pairs at the finest level on grids whose rows do not fill a workgroup (idle threads, a partial
last workgroup, workgroups past the last row), against the FP64 oracle with the tolerances of the sweep tests:
FP32 storage 2e-5; FP16 storage 3e-3 (2^-11 a rounding, with propagation over the colours)."""
import numpy as np
import pytest

import homo3d_amd

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a.astype(np.float64) - b) / np.linalg.norm(b)


@pytest.mark.parametrize("n", [20, 28, 40, 48, 56])
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("reverse", [False, True])
def test_sweep(orc, n, half, reverse):
    if half and n % 8:
        pytest.skip("packed FP16 fields need n % 8 == 0")
    print("sweep: n=%d half=%d reverse=%d" % (n, half, reverse), flush=True)
    hom = homo3d_amd.Homogenization(homo3d_amd.HomoConfig(reso=n, solver="pcg" if half else "mg", coarse_half=False))
    x = (homo3d_amd.randc_density(n, 7, 0.3, "none").astype(np.float64) ** 3).astype(np.float32)
    hom.update(x)
    mg = orc.MG(n, 10.0, 0.3)
    mg.set_density(x.astype(np.float64))
    rng = np.random.default_rng(n)
    u = (rng.standard_normal(hom.level_shape(0)) * 0.1).astype(np.float32)
    f = rng.standard_normal(hom.level_shape(0)).astype(np.float32)
    hom.set_field(0, 0, u)
    hom.set_field(0, 1, f)
    if half:
        u = u.astype(np.float16)
        hom.smooth16(1.0, reverse)
    else:
        hom.smooth(0, 1.0, reverse)
    got = hom.get_field(0, 0)
    for s in (0, 3, 5):
        ref = orc.gs_fine(n, mg.KE, mg.w, u[s].astype(np.float64), f[s].astype(np.float64), 1.0, reverse)
        assert rel(got[s], ref) < (3e-3 if half else 2e-5), s
