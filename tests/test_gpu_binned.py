"""One-shot backprojection of long lists (binned into tiles for the call) against the
same events in short lists (float atomics), summed in float64; and the cutting of a
plan's records into work items.

Non-negative values: a voxel of a short list gets at most a few hundred float
additions per list, 500 half-ulps = 3e-5 of its sum; a plan's term is resolved to 2^-50
of its item's largest, below 1e-9 of the image's largest voxel (a one-shot call's to
float64: test_gpu_binned_range.py holds every voxel to its own sum)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

REL, ABS = 500 * 2.0 ** -24, 1e-9


def _lors(n, seed, radius=150.0, axial=120.0):
    rng = np.random.default_rng(seed)
    phi = rng.uniform(0, 2 * np.pi, (n, 2))
    z = rng.uniform(-axial / 2, axial / 2, (n, 2))
    L = np.stack([radius * np.cos(phi[:, 0]), radius * np.sin(phi[:, 0]), z[:, 0], radius * np.cos(phi[:, 1]),
                  radius * np.sin(phi[:, 1]), z[:, 1], rng.normal(0, 50, n)], 1)
    L[0] = np.nan
    L[1, 2] = np.inf
    L[2, 3:6] = L[2, 0:3]
    L[3, :6] = [-150, 3.0, 1.0, 150, 3.0, 1.0]
    L[4, :6] = [3.0, -150, 1.0, 3.0, 150, 1.0]
    L[5, :6] = [-100, -100, 0.0, 100, 100, 0.0]
    L[6, :6] = [-100, 100, -5.0, 100, -100, 9.0]
    L[7, :6] = [0.0, 0.0, -60, 8.0, 0.0, 60]
    return torch.from_numpy(L.astype(np.float32)).cuda()


def _close(got, want):
    got = got.double()
    assert bool(torch.isfinite(got).all())
    err = (got - want).abs()
    print("largest error", float((err / want.clamp_min(1e-30)).max()), flush=True)
    assert bool((err <= REL * want + ABS * want.max()).all())


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("tof", [False, True])
@pytest.mark.parametrize("shape,voxel,n", [((48, 48, 24), (2.0, 2.0, 2.0), 90000), ((97, 31, 1), (2.0, 2.0, 2.0), 50000),
                                           ((33, 70, 41), (2.0, 2.0, 3.0), 70003), ((65, 64, 33), (2.0, 2.5, 2.0), 65537)])
def test_binned_equals_short_lists(shape, voxel, n, tof, mode):
    from srf_amd import ops
    L = _lors(n, shape[1])
    if not tof:
        L = L[:, :6].contiguous()
    v = torch.rand(n, generator=torch.Generator(device="cuda").manual_seed(3), device="cuda") + 0.1
    args = (list(shape), [0.7, -0.4, 1.1] + [a * b for a, b in zip(shape, voxel)], tof, 3.66, 649.2)
    step = 5000
    short = lambda w: sum(ops.backproject(L[k:k + step].contiguous(), None if w is None else w[k:k + step].contiguous(),
                                          *args, mode).double() for k in range(0, n, step))
    print("binned", shape, n, tof, mode, flush=True)
    _close(ops.backproject(L, v, *args, mode), short(v))
    _close(ops.backproject(L, None, *args, mode), short(None))
    p = v.clone()
    p[::7] = 0.0
    q = torch.where(p == 0, torch.zeros_like(v), v / p)
    _close(ops.backproject_ratio(L, v, p, 1, 0.0, *args, mode), short(q))


def test_accumulate_parts_and_capture():
    """accumulate = 1, a list longer than one part (2^21 events), and a captured call
    (atomics) of a list that is binned otherwise."""
    from srf_amd import ops
    from srf_amd._lib import check, lib, stream_handle
    shape, geom = (16, 16, 9), [0.0, 0.0, 0.0, 64.0, 64.0, 36.0]
    n = (1 << 21) + 12345
    L = _lors(n, 5)[:, :6].contiguous()
    grid = ops._grid(shape, geom)
    img = torch.ones((9, 16, 16), device="cuda")

    def add(lors, acc):
        check(lib().srf_backproject(lors.data_ptr(), lors.shape[0], 6, None, 0, None, grid, None, 0, acc, img.data_ptr(),
                                    stream_handle(img.device)), "srf_backproject")

    step = 20000
    want = torch.zeros((9, 16, 16), dtype=torch.float64, device="cuda")
    for k in range(0, n, step):
        want += ops.backproject(L[k:k + step].contiguous(), None, list(shape), geom, False, 0.0, 0.0, 0).double()
    add(L, 1)
    first = img.clone()
    # 20000 events put up to a few thousand additions on one of 2304 voxels
    bound = 20000 * 2.0 ** -24
    assert bool(((first.double() - 1 - want).abs() <= bound * want + 1e-6).all())
    add(L, 0)
    assert bool(((img.double() - want).abs() <= bound * want).all())
    m = 400000
    small = L[:m].contiguous()
    add(small, 0)
    eager = img.clone()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        add(small, 0)
    for _ in range(2):
        img.fill_(-1.0)
        g.replay()
        torch.cuda.synchronize()
        assert bool(((img - eager).abs() <= m * 2.0 ** -24 * eager).all())


@pytest.mark.parametrize("item", [256, 300, 1024, 8192])
@pytest.mark.parametrize("n", [20, 700, 30000, 250000])
def test_work_items(n, item):
    """A plan's items at most `item` records each, and its results those of the one-shot
    kernels on the same list (short lists; the sums' order differs)."""
    from srf_amd import ops
    shape, geom = (64, 48, 17), [0.0, 0.0, 0.0, 128.0, 96.0, 34.0]
    L = _lors(n, n)[8:].contiguous()
    n = L.shape[0]
    v = torch.rand(n, device="cuda") + 0.1
    img = torch.rand((17, 48, 64), device="cuda")
    plan = ops.Plan(L, shape, geom, True, 3.66, 649.2, item_records=item)
    info = plan.info()
    print("items", n, item, info, flush=True)
    assert info["items"] >= info["segments"] / item
    step = 5000
    want = sum(ops.backproject(L[k:k + step].contiguous(), v[k:k + step].contiguous(), list(shape), geom, True, 3.66, 649.2,
                               0).double() for k in range(0, n, step))
    _close(plan.backproject(v, 0), want)
    p = torch.cat([ops.project(L[k:k + step].contiguous(), img, list(shape), geom, True, 3.66, 649.2)
                   for k in range(0, n, step)])
    assert bool(((plan.project(img) - p).abs() <= 400 * 2.0 ** -24 * p + 1e-12).all())
    plan.close()
