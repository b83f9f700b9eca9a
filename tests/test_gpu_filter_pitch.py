"""The OC sensitivity filter in place on arrays with padded rows, in host and in device memory, by the staged
kernels and by the general one (radius 5): the live columns are those of unpadded arrays, the padding keeps its
values, and padded host arrays cost about what their bytes do."""
import ctypes
import time

import numpy as np
import pytest

import homo3d_amd

pytestmark = pytest.mark.gpu


def run(hom, sens, rho, pitch, radius, on_device):
    ptr = lambda a: a.ptr if on_device else ctypes.c_void_p(a.ctypes.data)
    rc = homo3d_amd.lib().homo3d_oc_filter(hom.handle, ptr(sens), ptr(rho), pitch, radius, 0, on_device)
    assert rc == homo3d_amd.HOMO3D_OK


@pytest.mark.parametrize("radius", [2.0, 5.0])
@pytest.mark.parametrize("on_device", [0, 1])
def test_padded_rows(radius, on_device):
    n, pitch = 32, 44
    print("padded filter: radius=%g on_device=%d" % (radius, on_device), flush=True)
    rng = np.random.default_rng(3)
    sens = -rng.uniform(0.1, 1.0, (n, n, pitch)).astype(np.float32)
    rho = rng.uniform(0.1, 1.0, (n, n, pitch)).astype(np.float32)
    hom = homo3d_amd.Homogenization(homo3d_amd.HomoConfig(reso=n, solver="none"))
    flat = np.ascontiguousarray(sens[:, :, :n])
    run(hom, flat, np.ascontiguousarray(rho[:, :, :n]), n, radius, 0)
    if on_device:
        d = homo3d_amd.DeviceBuffer.from_array(sens)
        run(hom, d, homo3d_amd.DeviceBuffer.from_array(rho), pitch, radius, 1)
        got = d.download().reshape(sens.shape)
    else:
        got = sens.copy()
        run(hom, got, rho, pitch, radius, 0)
    assert np.array_equal(got[:, :, :n], flat)
    assert np.array_equal(got[:, :, n:], sens[:, :, n:])


def test_padded_host_rows_are_not_copied_one_by_one():
    n, pitch = 128, 160
    print("padded filter, time", flush=True)
    hom = homo3d_amd.Homogenization(homo3d_amd.HomoConfig(reso=n, solver="none"))

    def best(p):
        sens = -np.ones((n, n, p), np.float32)
        rho = np.ones((n, n, p), np.float32)
        times = []
        for _ in range(6):
            t = time.perf_counter()
            run(hom, sens, rho, p, 2.0, 0)
            times.append(time.perf_counter() - t)
        return min(times[1:])

    # 1.25 times the bytes; row by row it was 100 times as long
    assert best(pitch) < 10 * best(n)
