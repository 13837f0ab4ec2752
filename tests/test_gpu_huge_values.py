"""Projections of images whose values come near float32's largest: a term is value times
weight, so that a projection overflows only where its own sum does (short lists, bundled
lists, point integrals).

Against float64 sums: float32 rounding of at most 3 x 200 terms."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

BOUND = 1200 * 2.0 ** -24


def _lors(n, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    phi = 2 * math.pi * torch.rand(n, generator=g, device="cuda")
    psi = phi + math.pi + 0.3 * torch.randn(n, generator=g, device="cuda")
    z = 40 * torch.rand(n, 2, generator=g, device="cuda") - 20
    return torch.stack([300 * torch.cos(phi), 300 * torch.sin(phi), z[:, 0], 300 * torch.cos(psi), 300 * torch.sin(psi),
                        z[:, 1], 20 * torch.randn(n, generator=g, device="cuda")], 1).contiguous()


@pytest.mark.parametrize("tof", [False, True])
@pytest.mark.parametrize("n", [500, 20000, 120000])
def test_projection_of_huge_values(n, tof):
    """The image times 2^100 projects to 2^100 times the image's projection (exact scaling)."""
    from srf_amd import ops
    shape, geom = [200, 190, 40], [0.0, 0.0, 0.0, 400.0, 380.0, 80.0]
    L = _lors(n, n)
    img = torch.rand((40, 190, 200), generator=torch.Generator(device="cuda").manual_seed(1), device="cuda") + 0.5
    p = ops.project(L, img, shape, geom, tof, 3.66, 649.2)
    big = ops.project(L, img * 2.0 ** 127, shape, geom, tof, 3.66, 649.2)
    assert bool(torch.isfinite(big).all())
    err = (big.double() / 2.0 ** 127 - p.double()).abs()
    print("largest", float(big.max()), float((err / p.double().clamp_min(1e-30)).max()), flush=True)
    assert bool((err <= BOUND * p.double()).all())


def test_point_integrals_of_huge_values():
    from srf_amd import ops
    shape, geom = [64, 60, 20], [0.0, 0.0, 0.0, 16.0, 15.0, 5.0]   # voxels of a quarter mm
    g = torch.Generator(device="cuda").manual_seed(2)
    phi = 2 * math.pi * torch.rand(300, generator=g, device="cuda")
    det = torch.stack([20 * torch.cos(phi), 20 * torch.sin(phi), torch.zeros_like(phi), phi], 1).contiguous()
    pts = ((torch.rand(400, 3, generator=g, device="cuda") - 0.5) * torch.tensor([10.0, 10.0, 4.0], device="cuda")).contiguous()
    img = torch.rand((20, 60, 64), generator=g, device="cuda") + 0.5
    for points in (pts, pts[:20].contiguous()):
        p = ops.point_integrals(det, points, img, shape, geom)
        big = ops.point_integrals(det, points, img * 2.0 ** 123, shape, geom)
        assert float(p.max()) * 2.0 ** 123 < 3e38 and bool(torch.isfinite(big).all())
        assert bool(((big.double() / 2.0 ** 123 - p.double()).abs() <= BOUND * p.double()).all())
