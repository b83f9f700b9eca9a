"""Sweeps of the small coarse levels (z-planes of 16 to 32 points an axis, a workgroup partly or more than
once filled) against the FP64 oracle, and whole V-cycles over every coarsest size, in which the bottom two levels
run as one launch (192 and 375 unknowns) or around the coarsest solve (648 and 1029), against the same cycle
made of the single operations."""
import numpy as np
import pytest

import homo3d_amd

pytestmark = pytest.mark.gpu


def design(n, seed, **kw):
    rho = homo3d_amd.randc_density(n, seed, 0.4, "none")
    x = (rho.astype(np.float64) ** 3).astype(np.float32)
    hom = homo3d_amd.Homogenization(homo3d_amd.HomoConfig(reso=n, **kw))
    hom.update(x)
    return hom, x


@pytest.mark.parametrize("n", [64, 40, 56])
@pytest.mark.parametrize("omega,reverse", [(1.0, False), (1.0, True), (0.8, False)])
def test_sweeps(orc, n, omega, reverse):
    print("sweeps: n=%d omega=%g reverse=%d" % (n, omega, reverse), flush=True)
    hom, _ = design(n, 5)
    rng = np.random.default_rng(n)
    for level in range(1, len(hom.sizes) - 1):
        m = hom.sizes[level]
        u = rng.standard_normal(hom.level_shape(level)).astype(np.float32)
        f = rng.standard_normal(hom.level_shape(level)).astype(np.float32)
        hom.set_field(level, 0, u)
        hom.set_field(level, 1, f)
        hom.smooth(level, omega, reverse)
        got = hom.get_field(level, 0)
        st = hom.stencil(level).astype(np.float64)
        for r in (0, 5):
            ref = orc.stencil_gs(m, st, u[r].astype(np.float64), f[r].astype(np.float64), omega, reverse)
            # a vertex sums 81 FP32 products and divides by its diagonal; eight colours pass the error on
            assert np.abs(got[r] - ref).max() <= 2e-5 * np.abs(ref).max(), (level, r)


@pytest.mark.parametrize("n", [16, 40, 24, 56])
@pytest.mark.parametrize("symmetric", [False, True])
def test_vcycle_is_its_parts(n, symmetric):
    print("vcycle: n=%d symmetric=%d" % (n, symmetric), flush=True)
    hom, _ = design(n, 7)
    hom.macro_rhs()
    f, zero = hom.get_field(0, 1), np.zeros(hom.level_shape(0), np.float32)
    hom.set_field(0, 0, zero)
    hom.vcycle(symmetric)
    got = [hom.get_field(level, 0) for level in range(len(hom.sizes))]
    hom.set_field(0, 0, zero)
    hom.set_field(0, 1, f)
    last = len(hom.sizes) - 1
    for level in range(last):
        hom.set_field(level, 0, np.zeros(hom.level_shape(level), np.float32))
        hom.smooth(level)
        hom.residual(level)
        hom.restrict(level + 1)
    hom.coarse_solve()
    for level in range(last - 1, -1, -1):
        hom.prolong(level)
        hom.smooth(level, reverse=symmetric)
    for level in range(last + 1):
        ref = hom.get_field(level, 0).astype(np.float64)
        # FP32 sums of 81 products in another order, through two sweeps a level and the coarsest solve's
        # condition (below 1e4 against the right-hand sides that occur)
        assert np.abs(got[level] - ref).max() <= 1e-4 * np.abs(ref).max(), level
