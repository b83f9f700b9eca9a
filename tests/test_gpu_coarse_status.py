"""Designs whose coarsest system is not positive definite: the solve names the first elimination step whose
pivot is not positive, wherever the step lies in its block of 32 and whichever block that is, and the handle
solves the next design as a fresh one does.  Coarsest systems of 192, 375, 648 and 1029 unknowns."""
import re

import numpy as np
import pytest

import homo3d_amd

pytestmark = pytest.mark.gpu


def first_bad_pivot(A):
    """Elimination without pivoting in FP64: the first step whose pivot is not positive, and how far each pivot
    up to it is from zero relative to its diagonal entry."""
    A = A.copy()
    scale, margin = np.abs(np.diag(A)).copy(), []
    for k in range(A.shape[0]):
        margin.append(abs(A[k, k]) / scale[k])
        if not A[k, k] > 0:
            return k, min(margin)
        A[k + 1:, k:] -= np.outer(A[k + 1:, k] / A[k, k], A[k, k:])
    return None, min(margin)


@pytest.mark.parametrize("n,plane", [(16, 0), (16, 9), (20, 10), (24, 14), (28, 6), (28, 22)])
def test_first_bad_pivot_is_reported(orc, n, plane):
    print("coarsest status: n=%d from plane %d" % (n, plane), flush=True)
    hom = homo3d_amd.Homogenization(homo3d_amd.HomoConfig(reso=n, coarse_half=False))
    good = (homo3d_amd.randc_density(n, 3, 0.4, "none").astype(np.float64) ** 3).astype(np.float32)
    bad = (0.2 + 0.8 * np.random.default_rng(n).random((n, n, n))).astype(np.float32)
    bad[plane:plane + 4] *= -1.5  # four planes of cells with negative stiffness
    hom.update(bad.reshape(-1))
    lc = len(hom.sizes) - 1
    A = orc.dense_from_stencil(hom.sizes[lc], hom.stencil(lc).astype(np.float64))
    k, margin = first_bad_pivot(0.5 * (A + A.T))
    # no pivot is so near zero that the order of the FP64 sums could change its sign
    assert k is not None and margin > 1e-9
    with pytest.raises(homo3d_amd.Homo3dError) as ei:
        hom.solve(1e-5, warm=False)
    assert ei.value.code == homo3d_amd.HOMO3D_DIVERGED
    assert re.search(r"pivot (\d+) of %d\b" % A.shape[0], str(ei.value)).group(1) == str(k)
    hom.update(good)
    C = hom.elasticMatrix(tol=1e-5, warm=False)
    fresh = homo3d_amd.Homogenization(homo3d_amd.HomoConfig(reso=n, coarse_half=False))
    fresh.update(good)
    assert np.array_equal(C, fresh.elasticMatrix(tol=1e-5, warm=False))
