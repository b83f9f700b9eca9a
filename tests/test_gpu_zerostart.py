"""The preconditioner's smoothing on grids whose rows do not fill a workgroup (idle threads, a partial last
workgroup): packed-FP16 sweeps, the zero-start sweeps whose passes leave their own-colour residuals, and those
residuals completed by the later colours' terms, at the finest and at coarse levels; FP32 sweeps and residuals
at 128^3 (rows as long as a wave).  Against the FP64 oracle.  Designs of x in [0.064, 1] and loads of unit size
keep u below some ten, far inside FP16."""
import numpy as np
import pytest

import homo3d_amd

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a.astype(np.float64) - b) / np.linalg.norm(b)


def design(n):
    rho = np.maximum(homo3d_amd.randc_density(n, 11, 0.3, "none").astype(np.float64), 0.4)
    return (rho ** 3).astype(np.float32)


def handle(n, coarse_half=False, solver="pcg"):
    hom = homo3d_amd.Homogenization(homo3d_amd.HomoConfig(reso=n, solver=solver, coarse_half=coarse_half,
                                                          fine_mfma=False))
    x = design(n)
    hom.update(x)
    return hom, 1e-9 + x.astype(np.float64)


def fields(hom, level, n, k):
    return (np.random.default_rng(n + i).standard_normal(hom.level_shape(level)).astype(np.float32) for i in range(k))


@pytest.mark.parametrize("n,omega", [(24, 1.0), (40, 1.0), (48, 0.8), (56, 1.0), (96, 1.0)])
def test_fine_presmooth(orc, n, omega):
    print("presmooth fp16: n=%d omega=%g" % (n, omega), flush=True)
    hom, w = handle(n)
    KE = orc.ke()
    f, u0 = fields(hom, 0, n, 2)
    hom.set_field(0, 1, f)
    hom.set_field(0, 0, u0)  # ignored
    hom.presmooth16(omega)
    u, r = hom.get_field(0, 0), hom.get_field(0, 2)
    zero = np.zeros(u.shape[1:])
    for s in range(6):
        # every new value is rounded to FP16 (2^-11) before later colours read it
        assert rel(u[s], orc.gs_fine(n, KE, w, zero, f[s].astype(np.float64), omega, False)) < 3e-3, s
        # the same u: 81 FP32 products a row
        assert rel(r[s], orc.residual(n, KE, w, u[s].astype(np.float64), f[s].astype(np.float64))) < 2e-6, s


@pytest.mark.parametrize("n", [40, 48, 56, 96])
@pytest.mark.parametrize("reverse", [False, True])
def test_fine_sweep_fp16(orc, n, reverse):
    print("sweep fp16: n=%d reverse=%d" % (n, reverse), flush=True)
    hom, w = handle(n)
    KE = orc.ke()
    f, u = fields(hom, 0, n, 2)
    hom.set_field(0, 1, f)
    hom.set_field(0, 0, u)
    hom.smooth16(1.0, reverse)
    got = hom.get_field(0, 0)
    u16 = u.astype(np.float16).astype(np.float64)
    for s in range(6):
        assert rel(got[s], orc.gs_fine(n, KE, w, u16[s], f[s].astype(np.float64), 1.0, reverse)) < 3e-3, s


@pytest.mark.parametrize("n,coarse_half", [(80, False), (96, True), (112, True)])
def test_coarse_presmooth(orc, n, coarse_half):
    print("coarse presmooth: level 1 of %d^3 half=%d" % (n, coarse_half), flush=True)
    hom, _ = handle(n, coarse_half)
    nc, st = hom.sizes[1], hom.stencil(1)
    f, u0 = fields(hom, 1, n, 2)
    hom.set_field(1, 1, f)
    hom.set_field(1, 0, u0)  # ignored
    hom.presmooth(1, 1.0)
    u, r = hom.get_field(1, 0), hom.get_field(1, 2)
    zero = np.zeros(u.shape[1:])
    for s in (0, 3, 5):
        # the tolerances of the coarse sweeps on levels that fill their workgroups
        assert rel(u[s], orc.stencil_gs(nc, st, zero, f[s].astype(np.float64), 1.0, False)) < 1e-5, s
        assert rel(r[s], orc.stencil_residual(nc, st, u[s].astype(np.float64), f[s].astype(np.float64))) < 1e-5, s


def test_small_levels_have_no_presmooth():
    hom, _ = handle(24)
    with pytest.raises(homo3d_amd.Homo3dError) as ei:
        hom.presmooth(1, 1.0)
    assert ei.value.code == homo3d_amd.HOMO3D_NO_SUPPORT


@pytest.mark.parametrize("reverse", [False, True])
def test_fp32_rows_of_a_wave(orc, reverse):
    n = 128
    print("fp32 sweep and residual: n=%d reverse=%d" % (n, reverse), flush=True)
    hom, w = handle(n, solver="mg")
    KE = orc.ke()
    f, u = fields(hom, 0, n, 2)
    u[:, :, 0] = 0
    hom.set_field(0, 1, f)
    hom.set_field(0, 0, u)
    hom.residual(0)
    r = hom.get_field(0, 2)
    hom.smooth(0, 1.0, reverse)
    got = hom.get_field(0, 0)
    s = 4
    # the tolerances of the other grids' FP32 sweeps and residuals
    assert rel(r[s], orc.residual(n, KE, w, u[s].astype(np.float64), f[s].astype(np.float64))) < 2e-6
    assert rel(got[s], orc.gs_fine(n, KE, w, u[s].astype(np.float64), f[s].astype(np.float64), 1.0, reverse)) < 2e-5
