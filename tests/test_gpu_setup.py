"""Galerkin stencils and the coarsest solve at every split of their kernels: level-1 grids of 8^3 to 56^3
(one direction a thread up to 32^3, nine up to 64^3), one to four coarser products, and coarsest systems of
192, 375 and 1029 unknowns (6, 12 and 33 blocks of 32, the last two partial), against the FP64 oracle."""
import numpy as np
import pytest

import homo3d_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [10, 16, 28, 40, 64, 112])
def test_stencils_and_coarse_solve(orc, n):
    print("setup: n=%d" % n, flush=True)
    rho = homo3d_amd.randc_density(n, 11, 0.4, "reflect3")
    x = (rho.astype(np.float64) ** 3).astype(np.float32)
    hom = homo3d_amd.Homogenization(homo3d_amd.HomoConfig(reso=n, coarse_half=False))
    hom.update(x)
    mg = orc.MG(n, 10.0, 0.3)
    mg.set_density(x.astype(np.float64))
    for level in range(1, len(hom.sizes)):
        if hom.sizes[level] > 28:
            continue  # 243 floats a vertex: the coarser levels are products of the finer ones
        ref = mg.stencil(level)
        # one FP32 rounding of the weights and one a level
        assert np.abs(hom.stencil(level) - ref).max() <= (level + 1) * 2.0 ** -24 * np.abs(ref).max(), level
    lc = len(hom.sizes) - 1
    nc = hom.sizes[lc]
    f = np.random.default_rng(n).standard_normal(hom.level_shape(lc)).astype(np.float32)
    hom.set_field(lc, 1, f)
    hom.coarse_solve()
    u = hom.get_field(lc, 0).astype(np.float64)
    A = orc.dense_from_stencil(nc, hom.stencil(lc).astype(np.float64))
    A = 0.5 * (A + A.T)
    for s in range(6):
        ref = np.linalg.solve(A, f[s].astype(np.float64).T.reshape(-1)).reshape(-1, 3).T
        # the same FP64 system (condition below 1e5), the solution rounded to FP32
        assert np.abs(u[s] - ref).max() <= 2.0 ** -23 * np.abs(ref).max(), s
