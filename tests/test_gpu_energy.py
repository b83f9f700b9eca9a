"""C^H and sensitivity of given fields on grids whose last energy tiles (32 x 4 x 2 cells) are partial,
with an odd half-size, and at a material other than the default, against the FP64 oracle."""
import numpy as np
import pytest

import homo3d_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,E,nu", [(8, 10.0, 0.3), (10, 10.0, 0.3), (32, 1.0, 0.0), (40, 3.0, -0.2)])
def test_energies_of_given_fields(orc, n, E, nu):
    print("energies: n=%d E=%g nu=%g" % (n, E, nu), flush=True)
    rng = np.random.default_rng(n)
    hom = homo3d_amd.Homogenization(homo3d_amd.HomoConfig(reso=n, youngsModulu=E, poissonRatio=nu))
    x = rng.uniform(0.01, 1.0, n ** 3).astype(np.float32)
    hom.update(x)
    chi = rng.uniform(-0.5, 0.5, (6, 3, n ** 3)).astype(np.float32)
    hom.set_field(0, homo3d_amd.FIELD_U, chi)
    KE = orc.ke(E, nu)
    w = 1e-9 + x.astype(np.float64)
    C, Cref = hom.elasticMatrix(solve=False), orc.elastic_matrix(n, KE, w, chi.astype(np.float64))
    # a cell's energies carry some 40 FP32 roundings of the size of its largest energy, of random signs
    # and averaged over the cells; the sensitivity holds one cell's
    assert np.abs(C - Cref).max() <= 2e-6 * np.abs(Cref).max()
    dC = rng.uniform(-1.0, 1.0, (6, 6)).astype(np.float32)
    s, sref = hom.Sensitivity(dC), orc.sensitivity(n, KE, chi.astype(np.float64), dC.astype(np.float64))
    assert np.abs(s - sref).max() <= 40 * 2.0 ** -24 * np.abs(sref).max()
    pitched = hom.Sensitivity(dC, pitchT=n + 3).reshape(n, n, n + 3)
    assert np.array_equal(pitched[:, :, :n].ravel(), s) and not pitched[:, :, n:].any()
