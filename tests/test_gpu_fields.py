"""The staged filter kernels at the edges of their tiles (32 x 8 x 8 cells) and of the grid, for every
half-width they take and the general kernel beyond (h = 4), and the elementwise maps on unaligned and
pitched device arrays, against the FP64 oracles."""
import ctypes

import numpy as np
import pytest

import homo3d_amd
from oracle import filter_oracle as fo

pytestmark = pytest.mark.gpu


def handle(n):
    return homo3d_amd.Homogenization(homo3d_amd.HomoConfig(reso=n, solver="none"))


def close(got, want, ulps):
    """ulps: FP32 roundings (2^-24 each) that the result carries, relative to the largest entry."""
    return np.abs(np.asarray(got, np.float64) - want).max() <= ulps * 2.0 ** -24 * np.abs(want).max()


@pytest.mark.parametrize("n,radius", [(5, 2.0), (8, 1.0), (31, 1.5), (33, 2.3), (40, 3.4), (9, 3.0), (12, 4.2)])
@pytest.mark.parametrize("periodic", [False, True])
def test_filters(orc, n, radius, periodic):
    print("filters: n=%d radius=%g periodic=%d" % (n, radius, periodic), flush=True)
    rng = np.random.default_rng(n)
    a = rng.uniform(0.1, 1.0, (n, n, n)).astype(np.float32)
    g = rng.uniform(-1.0, 1.0, (n, n, n)).astype(np.float32)
    hom = handle(n)
    for kern in ("spline4", "linear"):
        want, _ = fo.conv(a, radius, periodic, kern)
        # FP32 weights (half an ulp each in numerator and denominator) and one rounding of the result
        assert close(hom.density_filter(a, radius, kern, periodic).reshape(a.shape), want, 4), kern
        want = fo.conv_backward(g, radius, periodic, kern)
        # the adjoint also divides by FP32-rounded weight sums; the signed terms cancel, so the rounding is
        # measured against the sum of their magnitudes (at most 4 times the largest entry here)
        assert close(hom.density_filter(g, radius, kern, periodic, backward=True).reshape(a.shape), want, 16), kern
    want = orc.oc_filter(n, g.ravel().astype(np.float64), a.ravel().astype(np.float64), radius, periodic)
    got = homo3d_amd.OCOptimizer(hom).filterSens(g, a, radius, periodic)
    assert close(got, want, 64)  # divided by rho >= 0.1


@pytest.mark.parametrize("n,pitch,shift", [(8, 8, 0), (8, 8, 1), (7, 7, 0), (33, 40, 0), (65, 65, 3)])
def test_maps_on_device_arrays(n, pitch, shift):
    print("maps: n=%d pitch=%d shift=%d" % (n, pitch, shift), flush=True)
    rng = np.random.default_rng(n)
    L, hom = homo3d_amd.lib(), handle(n)
    elems = pitch * n * n
    full = rng.uniform(0.05, 1.0, (3, elems + shift)).astype(np.float32)
    bufs = [homo3d_amd.DeviceBuffer.from_array(f) for f in full]
    ptr = [ctypes.c_void_p(b.value + 4 * shift) for b in bufs]
    view = [f[shift:].reshape(n, n, pitch) for f in full]
    live = (slice(None), slice(None), slice(0, n))

    def result(want, ulps):
        out = bufs[2].download()
        got = out[shift:].reshape(n, n, pitch)
        assert np.array_equal(out[:shift], full[2][:shift])
        assert np.array_equal(got[:, :, n:], view[2][:, :, n:])  # padding keeps its values
        assert close(got[live], want, ulps)

    a, b = view[0][live].astype(np.float64), view[1][live].astype(np.float64)
    assert L.homo3d_projection(hom.handle, ptr[0], None, ptr[2], pitch, 30.0, 0.5, 0, 1) == 0
    result(fo.sgm(a), 2)
    assert L.homo3d_projection(hom.handle, ptr[0], ptr[1], ptr[2], pitch, 30.0, 0.5, 1, 1) == 0
    result(fo.sgm_backward(b, a), 2)
    assert L.homo3d_density_pow(hom.handle, ptr[0], ptr[2], pitch, 3.0, 1) == 0
    result(a ** 3, 4)
    assert L.homo3d_density_pow_grad(hom.handle, ptr[0], ptr[1], ptr[2], pitch, 3.0, 1) == 0
    result(3 * a * a * b, 6)
    assert L.homo3d_density_filter(hom.handle, ptr[0], ptr[2], pitch, 2.0, 0, 0, 0, 1) == 0
    result(fo.conv(a, 2.0)[0], 4)


@pytest.mark.parametrize("n", [20, 28, 72])
@pytest.mark.parametrize("sym", ["reflect3", "reflect6", "rotate3"])
def test_symmetrize(orc, n, sym):
    """Orbits across partial workgroups, bit for bit (the FP64 sums run in the group's order)."""
    print("symmetrize: n=%d %s" % (n, sym), flush=True)
    hom = homo3d_amd.Homogenization(homo3d_amd.HomoConfig(reso=n, solver="none"))
    f = np.random.default_rng(n).standard_normal(n ** 3).astype(np.float32)
    assert np.array_equal(hom.symmetrize(f, sym), orc.symmetrize(n, f, sym))
