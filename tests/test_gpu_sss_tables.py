"""The SSS kernels in the layout for bins in any order, at small and odd numbers of
detectors, points (groups of 16) and bins, an index outside the table, and the point line
integrals over the copies and without them.  (Both layouts at the edges of their groups,
workgroups and lanes: test_gpu_sss_orders.py.)

Bin sums against float64 with the whole-degree angle of each pair taken from the
float32 cosine the path forms (unit vectors and three fused multiply-adds), so that no
pair sits on another side of a degree: what is left is float32
rounding, 1e-5 of the terms' sum as in the other tests, and what lies below float32's
normal range (2^-126; pairs far outside the energy window)."""
import math

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _tables():
    from srf_amd.sss import energy_tables
    return energy_tables(400.0, 650.0, 0.15, True)


def _fma32(a, b, c):
    return (a.double() * b.double() + c.double()).float()


def _fma64(x, y, z):
    return x * x + (y * y + z * z)                         # squares of floats are exact in double


def _sum64(det, pts, em, mu, bins, tab):
    v = det[:, None, :3] - pts[None, :, :3]
    r2 = v[..., 0] * v[..., 0] + v[..., 1] * v[..., 1] + v[..., 2] * v[..., 2]
    u = v * (1.0 / torch.sqrt(r2))[..., None]
    q = u.double()
    half = (0.5 * (1.0 - _fma64(q[..., 0], q[..., 1], q[..., 2]))).float()
    u = _fma32(u, half[..., None], u)
    a, b = bins[:, 0].long(), bins[:, 1].long()
    x = -_fma32(u[a, :, 0], u[b, :, 0], _fma32(u[a, :, 1], u[b, :, 1], u[a, :, 2] * u[b, :, 2]))
    k = torch.clamp((torch.acos(x.clamp(-1, 1).double()) * 57.295779513082323).long(), 0, 180)
    v, d = v.double(), det.double()
    r = v.norm(dim=2)
    g = (v[..., 0] * torch.cos(d[:, 3])[:, None] + v[..., 1] * torch.sin(d[:, 3])[:, None]) / r ** 3
    t = torch.from_numpy(tab).cuda().double()
    rr = t[k]
    E, M = em.double(), mu.double()
    I = torch.exp(-(M[a] + M[b] * rr)) * E[a] + torch.exp(-(M[a] * rr + M[b])) * E[b]
    return g[a] * g[b] * t[181 + k] * t[362 + k] * pts[None, :, 3].double() * I


@pytest.mark.parametrize("nd,ns,nb", [(8, 1, 1), (8, 2, 63), (16, 15, 64), (16, 16, 65), (40, 17, 200), (64, 300, 130),
                                      (64, 1025, 70), (32, 2600, 5000), (8200, 15, 300), (8200, 16, 64), (8200, 18, 300),
                                      (8201, 37, 1000), (8200, 600, 129)])
def test_bin_sums(nd, ns, nb):
    from srf_amd._lib import check, lib, stream_handle
    g = torch.Generator(device="cuda").manual_seed(nd + 7 * ns)
    rnd = lambda *s: torch.rand(s, generator=g, device="cuda")
    phi = 2 * math.pi * rnd(nd)
    det = torch.stack([424 * torch.cos(phi), 424 * torch.sin(phi), 300 * rnd(nd) - 150, phi], 1).contiguous()
    pts = torch.cat([240 * rnd(ns, 3) - 120, 0.005 + 0.01 * rnd(ns, 1)], 1)
    if ns > 16:
        pts[5, 3] = 0.0                                   # skipped, whatever its rows hold
    pts = pts.contiguous()
    em, mu = 50 * rnd(nd, ns), 3 * rnd(nd, ns)
    if ns > 16:
        em[:, 5] = float("nan")
    bins = torch.randint(0, nd, (nb, 2), generator=g, device="cuda", dtype=torch.int32)
    s = torch.cuda.current_stream().cuda_stream
    L = lib()
    need = L.srf_sss_rows_bytes(nd, ns)
    rows = torch.empty(need // 4 + 4, device="cuda")
    tab = _tables()
    t = torch.from_numpy(tab).cuda()
    out = torch.full((nb,), -1.0, device="cuda")
    print("sss", nd, ns, nb, flush=True)
    check(L.srf_sss_prepare(det.data_ptr(), nd, pts.data_ptr(), ns, em.data_ptr(), mu.data_ptr(), rows.data_ptr(), need,
                            stream_handle(out.device)), "prepare")
    check(L.srf_sss_sinogram(rows.data_ptr(), nd, pts.data_ptr(), ns, bins.data_ptr(), nb, t.data_ptr(), 2.0,
                             out.data_ptr(), s), "sinogram")
    terms = _sum64(det, pts, torch.nan_to_num(em), mu, bins, tab)
    want = 2.0 * terms.sum(1)
    assert bool(((out.double() - want).abs() <= 1e-5 * 2.0 * terms.abs().sum(1) + 2.0 ** -126).all())
    if nb > 2:
        bad = bins.clone()
        bad[1, 0], bad[2, 1] = -1, nd
        check(L.srf_sss_sinogram(rows.data_ptr(), nd, pts.data_ptr(), ns, bad.data_ptr(), nb, t.data_ptr(), 2.0,
                                 out.data_ptr(), s), "sinogram")
        assert bool(torch.isnan(out[1:3]).all()) and int(torch.isnan(out).sum()) == 2


@pytest.mark.parametrize("nd,ns", [(3, 1), (70, 255), (66, 257), (130, 600)])
@pytest.mark.parametrize("shape,size", [((40, 33, 17), (80.0, 66.0, 34.0)), ((32, 40, 20), (80.0, 100.0, 60.0))])
def test_point_integrals_equal_projector(nd, ns, shape, size):
    """Against srf_project along the same LORs, times L^2 / dx^2 (float32 products: 1e-6
    and the two summation orders, 3 x 40 terms), eager (over the copies from 64 workgroups
    on) and captured (without them)."""
    from srf_amd import ops
    from srf_amd._lib import check, lib, stream_handle
    g = torch.Generator(device="cuda").manual_seed(ns)
    rnd = lambda *s: torch.rand(s, generator=g, device="cuda")
    phi = 2 * math.pi * rnd(nd)
    det = torch.stack([70 * torch.cos(phi), 70 * torch.sin(phi), 50 * rnd(nd) - 25, phi], 1).contiguous()
    pts = torch.cat([(rnd(ns, 3) - 0.5) * torch.tensor(size, device="cuda"), rnd(ns, 1)], 1).contiguous()
    if nd > 3:
        det[1, 0] = float("nan")
    img = rnd(shape[2], shape[1], shape[0])
    geom = [0.0, 0.0, 0.0] + list(size)
    lors = torch.cat([det[:, None, :3].expand(nd, ns, 3), pts[None, :, :3].expand(nd, ns, 3)], 2).reshape(-1, 6).contiguous()
    L2 = ((lors[:, 3:6].double() - lors[:, :3].double()) ** 2).sum(1) / (size[0] / shape[0]) ** 2
    want = (ops.project(lors, img, list(shape), geom, False, 0.0, 0.0).double() * L2).reshape(nd, ns)
    out = torch.full((nd, ns), -1.0, device="cuda")

    def call():
        check(lib().srf_sss_integrals(det.data_ptr(), nd, pts.data_ptr(), ns, 4, img.data_ptr(), ops._grid(shape, geom),
                                      out.data_ptr(), stream_handle(out.device)), "srf_sss_integrals")

    call()
    graph = torch.cuda.CUDAGraph()
    eager = out.clone()
    with torch.cuda.graph(graph):
        call()
    out.fill_(-1.0)
    graph.replay()
    torch.cuda.synchronize()
    for got in (eager, out):
        assert torch.equal(torch.isnan(got), torch.isnan(want))
        ok = ~torch.isnan(want)
        assert bool(((got.double() - want).abs() <= (1e-6 + 240 * 2.0 ** -24) * want.abs())[ok].all())


def test_rejected_arguments():
    from srf_amd import ops
    from srf_amd._lib import lib
    x = torch.zeros(64, device="cuda")
    grid = ops._grid((2, 2, 2), [0.0, 0.0, 0.0, 4.0, 4.0, 4.0])
    p = x.data_ptr()
    assert lib().srf_sss_integrals(p, 0, p, 1, 4, p, grid, p, None) == -1
    assert lib().srf_sss_integrals(p, 1, p, 1, 2, p, grid, p, None) == -1
    assert lib().srf_sss_integrals(None, 1, p, 1, 4, p, grid, p, None) == -1
