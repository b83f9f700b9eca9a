"""GPU test of the weight gradient with four tiles of output channels on rows of 32 and 64 voxels (106 and 117 KB
of LDS a workgroup), against the FP64 oracle with the tolerances of the other gradient tests."""
import pytest

from tests.test_gpu_netgrad import test_gradient as check_gradient

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("g", [32, 64])
def test_four_output_tiles(g):
    check_gradient(g, 1, 64, 1)
