"""The bundled projector (srf_project on long lists; 1, 2 and 4 wavefronts per bundle)
against the one-event-per-lane path on the same events: split into lists below the
bundling size (2e7 slabs), a list runs k_gather, whose voxel indexing the digest
tests pin.  Both evaluate the same slabs
with the same fractions and differ in the order of the sums only (k_gather's lanes
sum runs of slabs): float32 sums of at most 3 x 210 non-negative terms agree to
1260 half-ulps, 7.5e-5 relative.  Also non-finite and skipped LORs among the others,
LORs along the axes, ties |dx| == |dy|, odd strides, and a captured call (which keeps
the unsorted path)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

BOUND = 1260 * 2.0 ** -24


def _lors(n, seed, radius=150.0, axial=120.0):
    rng = np.random.default_rng(seed)
    phi = rng.uniform(0, 2 * np.pi, (n, 2))
    z = rng.uniform(-axial / 2, axial / 2, (n, 2))
    L = np.stack([radius * np.cos(phi[:, 0]), radius * np.sin(phi[:, 0]), z[:, 0], radius * np.cos(phi[:, 1]),
                  radius * np.sin(phi[:, 1]), z[:, 1], rng.normal(0, 50, n)], 1)
    L[0] = np.nan
    L[1, 2] = np.inf
    L[2, 3:6] = L[2, 0:3]                                   # no extent
    L[3, :6] = [-150, 3.0, 1.0, 150, 3.0, 1.0]              # along x, y
    L[4, :6] = [3.0, -150, 1.0, 3.0, 150, 1.0]
    L[5, :6] = [-100, -100, 0.0, 100, 100, 0.0]             # ties of the dominant axis
    L[6, :6] = [-100, 100, -5.0, 100, -100, 9.0]
    L[7, :6] = [0.0, 0.0, -60, 8.0, 0.0, 60]                # steep
    L[8, :6] = [-150, 400, 0, 150, 400, 0]                  # outside the image
    L[9, :6] = [-20, 1.0, 0.5, 10.0, 1.0, 0.5]              # ends inside it
    return L.astype(np.float32)


@pytest.mark.parametrize("tof", [False, True])
@pytest.mark.parametrize("shape,voxel,n", [((210, 200, 41), (1.0, 1.0, 2.0), 100077), ((130, 130, 80), (2.0, 2.0, 2.0), 160001),
                                           ((97, 70, 199), (2.0, 2.0, 1.5), 300000), ((128, 64, 70), (2.0, 2.5, 2.0), 350003),
                                           ((1, 200, 2000), (2.0, 2.0, 0.25), 262145)])
def test_bundled_equals_short_lists(shape, voxel, n, tof):
    from srf_amd import ops
    L = torch.from_numpy(_lors(n, shape[0])).cuda()
    if not tof:
        L = L[:, :6].contiguous()
    g = torch.Generator(device="cuda").manual_seed(shape[1])
    img = torch.rand((shape[2], shape[1], shape[0]), generator=g, device="cuda")
    geom = [0.7, -0.4, 1.1] + [n_ * v for n_, v in zip(shape, voxel)]
    args = (list(shape), geom, tof, 3.66, 649.2)
    print("bundle", shape, voxel, tof, flush=True)
    got = ops.project(L, img, *args)
    want = torch.cat([ops.project(L[k:k + 40000].contiguous(), img, *args) for k in range(0, n, 40000)])
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and int(torch.isnan(got).sum()) == 2
    ok = ~torch.isnan(want)
    assert torch.equal(got[ok] == 0, want[ok] == 0)
    assert bool(((got - want).abs() <= BOUND * want.abs())[ok].all())
    if n == 100077:
        wide = torch.cat([L, torch.zeros((n, 4), device="cuda")], 1).contiguous()
        tv = L[:, 6].contiguous() if tof else None
        assert torch.equal(torch.nan_to_num(ops.project(wide, img, *args, tv), nan=-1.0),
                           torch.nan_to_num(got, nan=-1.0))


def test_captured_call_and_short_list_lanes():
    from srf_amd import ops
    shape, geom = [210, 200, 41], [0.0, 0.0, 0.0, 210.0, 200.0, 82.0]
    L = torch.from_numpy(_lors(100005, 3)[10:]).cuda()
    img = torch.rand((41, 200, 210), device="cuda")
    eager = ops.project(L, img, shape, geom, True, 3.66, 649.2)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = ops.project(L, img, shape, geom, True, 3.66, 649.2)
    for _ in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert bool(((out - eager).abs() <= BOUND * eager).all())
    # 1 to 16 lanes per event, whole and partly filled blocks
    for n in (1, 3, 16, 255, 4096, 8193, 20000, 40001, 70000):
        p = ops.project(L[:n].contiguous(), img, shape, geom, True, 3.66, 649.2)
        assert bool(((p - eager[:n]).abs() <= BOUND * eager[:n]).all()), n
