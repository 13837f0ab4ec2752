"""Projector on several images: what one image at a time takes, the batch takes."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B", [1, 2, 3])
def test_images_by_their_voxel_count(B):
    """An image is read as voxel count says, one by one or as a batch."""
    from siddon_ref import random_cylinder_lors
    from srf_amd.autograd import Projector
    L = torch.from_numpy(np.ascontiguousarray(random_cylinder_lors(500, 150.0, 80.0, 1))).cuda()
    P = Projector(L, (24, 20, 8), [0.0, 0.0, 0.0], [96.0, 80.0, 32.0])
    x = torch.rand((B, 20, 24, 8), device="cuda")
    assert torch.equal(P(x), torch.stack([P(x[b]) for b in range(B)]))
    for bad in (torch.rand((B, 24, 20, 9), device="cuda"), torch.rand((B, 24, 20, 8), device="cuda").double()):
        with pytest.raises(ValueError):
            P(bad)
