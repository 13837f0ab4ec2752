"""The SSS bin sums in both row layouts (any order, sinogram order) at their edges: points
per group (4, 16; partial last groups), bins per workgroup (1024), points split over
workgroups, and the change from 64 to 16 lanes per bin (below 256 points, from 8192 bins
on).  Reference and bound as in test_gpu_sss_tables.py."""
import math

import pytest
import torch

from test_gpu_sss_tables import _sum64, _tables

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ordered", [False, True])
@pytest.mark.parametrize("nd,ns,nb", [(64, 1, 1), (64, 15, 1023), (64, 16, 1024), (64, 17, 1025), (40, 31, 3), (40, 33, 4),
                                      (40, 300, 1025), (8200, 18, 300), (300, 33, 65541), (70, 255, 50),
                                      (70, 256, 51), (70, 257, 8191), (70, 273, 8192), (16, 5, 65536),
                                      (32, 2600, 5000)])
def test_bin_sums(nd, ns, nb, ordered):
    from srf_amd._lib import check, lib, stream_handle
    g = torch.Generator(device="cuda").manual_seed(3 * nd + 7 * ns)
    rnd = lambda *s: torch.rand(s, generator=g, device="cuda")
    phi = 2 * math.pi * rnd(nd)
    det = torch.stack([424 * torch.cos(phi), 424 * torch.sin(phi), 300 * rnd(nd) - 150, phi], 1).contiguous()
    pts = torch.cat([240 * rnd(ns, 3) - 120, 0.005 + 0.01 * rnd(ns, 1)], 1)
    em, mu = 50 * rnd(nd, ns), 3 * rnd(nd, ns)
    if ns > 8:
        pts[ns - 3, 3] = 0.0                              # skipped, whatever its rows hold
        em[:, ns - 3] = float("nan")
    pts = pts.contiguous()
    bins = torch.randint(0, nd, (nb, 2), generator=g, device="cuda", dtype=torch.int32)
    L, s = lib(), stream_handle(det.device)
    prepare = L.srf_sss_prepare_ordered if ordered else L.srf_sss_prepare
    sinogram = L.srf_sss_sinogram_ordered if ordered else L.srf_sss_sinogram
    need = L.srf_sss_rows_bytes(nd, ns)
    rows = torch.full((need // 4 + 64,), -7.0, device="cuda")
    tab = _tables()
    t = torch.from_numpy(tab).cuda()
    out = torch.full((nb,), -1.0, device="cuda")
    print("sss", nd, ns, nb, ordered, flush=True)
    check(prepare(det.data_ptr(), nd, pts.data_ptr(), ns, em.data_ptr(), mu.data_ptr(), rows.data_ptr(), need, s), "prepare")
    assert bool((rows[need // 4:] == -7.0).all())         # nothing past the workspace
    check(sinogram(rows.data_ptr(), nd, pts.data_ptr(), ns, bins.data_ptr(), nb, t.data_ptr(), 2.0, out.data_ptr(), s),
          "sinogram")
    terms = _sum64(det, pts, torch.nan_to_num(em), mu, bins, tab)
    assert bool(((out.double() - 2.0 * terms.sum(1)).abs() <= 1e-5 * 2.0 * terms.abs().sum(1) + 2.0 ** -126).all())
    if nb > 2:
        bins[1, 0], bins[2, 1] = -1, nd
        check(sinogram(rows.data_ptr(), nd, pts.data_ptr(), ns, bins.data_ptr(), nb, t.data_ptr(), 2.0, out.data_ptr(), s),
              "sinogram")
        assert bool(torch.isnan(out[1:3]).all()) and int(torch.isnan(out).sum()) == 2


def test_rejected_arguments():
    from srf_amd._lib import lib
    x = torch.zeros(4096, device="cuda")
    p, L = x.data_ptr(), lib()
    for prepare in (L.srf_sss_prepare, L.srf_sss_prepare_ordered):
        assert prepare(p, 0, p, 1, p, p, p, 4096, None) == -1
        assert prepare(p, 2, p, 2, p, p, p, 127, None) == -4
        assert prepare(p, 2, p, 2, p, p, p + 4, 4096, None) == -1
    for sinogram in (L.srf_sss_sinogram, L.srf_sss_sinogram_ordered):
        assert sinogram(p, 1, p, 1, None, 1, p, 1.0, p, None) == -1
        assert sinogram(p, 1, p, 1, p, -1, p, 1.0, p, None) == -1
        assert sinogram(p, 1, p, 1, p, 0, p, 1.0, p, None) == 0
