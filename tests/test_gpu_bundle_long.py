"""The bundled projector on images that fit an XCD's L2, whose lists are bundled from 6e7 slabs
on: the comparison of test_gpu_bundle.py on longer lists."""
import pytest

import test_gpu_bundle as tb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tof", [False, True])
@pytest.mark.parametrize("shape,voxel,n", [((128, 64, 70), (2.0, 2.5, 2.0), 500003), ((1, 200, 2000), (2.0, 2.0, 0.25), 320001)])
def test_bundled_equals_short_lists(shape, voxel, n, tof):
    tb.test_bundled_equals_short_lists(shape, voxel, n, tof)
