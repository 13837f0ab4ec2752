"""One-shot backprojection on a grid whose events have many segments: parts by segments, so
that the scratch of a call, and what the pool keeps of it, stay near 4 GB."""
import pytest
import torch

pytestmark = pytest.mark.gpu

REL = 500 * 2.0 ** -24


def test_scratch_is_bounded_by_segments():
    from srf_amd import ops
    # a long grid: a line crosses its 64 tiles along x and some of the others
    shape, geom = [2048, 64, 64], [0.0, 0.0, 0.0, 2048.0, 64.0, 64.0]
    n = 1200000
    g = torch.Generator(device="cuda").manual_seed(4)
    yz = 60 * torch.rand(n, 4, generator=g, device="cuda") - 30
    x = torch.full((n, 1), 1200.0, device="cuda")
    L = torch.cat([-x, yz[:, :2], x, yz[:, 2:]], 1).contiguous()
    torch.cuda.synchronize()
    ops.trim_plan_pool(0)
    torch.cuda.empty_cache()
    free0 = torch.cuda.mem_get_info()[0]
    img = ops.backproject(L, None, shape, geom, False, 0.0, 0.0, 0)
    torch.cuda.synchronize()
    taken = free0 - torch.cuda.mem_get_info()[0] - img.numel() * 4
    print("scratch kept", taken / 1e9, flush=True)
    assert 3e9 < taken < 5e9     # about 4 GB; the whole list would take 8
    ops.trim_plan_pool(0)
    assert free0 - torch.cuda.mem_get_info()[0] < 0.5e9
    # against plans of pieces (fixed point; no TOF, so that they hold every term)
    want = torch.zeros((64, 64, 2048), dtype=torch.float64, device="cuda")
    for k in range(0, n, 300000):
        p = ops.Plan(L[k:k + 300000].contiguous(), shape, geom, False)
        want += p.backproject(None, 0).double()
        p.close()
    assert bool(((img.double() - want).abs() <= REL * want + 1e-9 * want.max()).all())
    ops.trim_plan_pool(0)
