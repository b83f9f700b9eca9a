"""The benchmark's bytes of a Gauss-Seidel launch: a pair of the eight colours on every grid."""
import pytest

import bench


@pytest.mark.parametrize("n", [32, 80, 192, 256])
def test_gauss_seidel_launch_is_a_colour_pair(n):
    N, R = n ** 3, 6
    sweep = N * (3 * R * (2 * 2 + 4) + 4)  # packed-FP16 z read and written, FP32 f and weights read
    assert bench.kernel_bytes("fine_gs", n) == sweep / 4
    # a quarter of the vertices updated, the whole field and every weight read
    assert bench.gs_pair_must_read(n) == N * (3 * R * 2 + 4) + N / 4 * 3 * R * (4 + 2)
