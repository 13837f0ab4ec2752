"""Several images in one call (srf_plan_project_batch: two images share a march;
plan_backproject_batch): bit-identical to the single calls for every count, with and
without TOF, on anisotropic voxels, for values that need the exponent
bands or are not finite in one image of a pair only, under capture, and through
autograd."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _plan(shape, voxel, n, tof, seed=1):
    from siddon_ref import random_cylinder_lors
    from srf_amd import ops
    L = random_cylinder_lors(n, 150.0, 80.0, seed, tof_sigma=25.48 if tof else None)
    if n > 3:
        L[3, 0] = np.nan
    geom = [0.0, 0.0, 0.0] + [a * b for a, b in zip(shape, voxel)]
    return ops.Plan(torch.from_numpy(np.ascontiguousarray(L)).cuda(), shape, geom, tof, 3.66, 649.2), n


@pytest.mark.parametrize("tof", [False, True])
@pytest.mark.parametrize("shape,voxel,n", [((48, 48, 24), (2.0, 2.0, 2.0), 30000), ((33, 65, 9), (2.0, 2.0, 3.0), 5001),
                                           ((40, 31, 17), (2.0, 2.5, 2.0), 2000), ((16, 16, 8), (4.0, 4.0, 4.0), 1)])
def test_batch_equals_single_calls(shape, voxel, n, tof):
    plan, n = _plan(shape, voxel, n, tof)
    g = torch.Generator(device="cuda").manual_seed(7)
    from srf_amd import ops
    for B in (1, 2, 3, 4, 5, 7, 8):
        print("multi", shape, n, tof, B, flush=True)
        x = torch.rand((B, shape[2], shape[1], shape[0]), generator=g, device="cuda")
        p = plan.project_batch(x)
        for b in range(B):
            assert torch.equal(torch.nan_to_num(p[b], nan=-1.0), torch.nan_to_num(plan.project(x[b]), nan=-1.0))
        v = torch.rand((B, n), generator=g, device="cuda") * 10.0 ** torch.arange(B, device="cuda")[:, None]
        if B > 2 and n > 100:
            v[1, ::9] *= 1e12            # exponent bands in one image of a pair
            v[2, 7] = float("nan")       # float tiles in another
            v[0, :] = 0.0
        for mode in (0, 1):
            q = ops.plan_backproject_batch(plan.handle, v, n, plan.shape, mode)
            for b in range(B):
                one = plan.backproject(v[b].contiguous(), mode)
                if b == 2 and B > 2 and n > 100:   # float atomics: an order of their own
                    assert torch.equal(torch.isnan(q[b]), torch.isnan(one))
                    ok = ~torch.isnan(one)
                    assert bool(((q[b] - one).abs() <= 1e-4 * one.abs() + 1e-6 * one[ok].abs().max())[ok].all())
                else:
                    assert torch.equal(q[b], one)
    plan.close()


def test_capture_and_autograd():
    from siddon_ref import random_cylinder_lors
    from srf_amd.autograd import Projector
    shape, size = (48, 40, 24), [96.0, 80.0, 48.0]
    L = torch.from_numpy(random_cylinder_lors(20000, 150.0, 80.0, 5, tof_sigma=25.48)).cuda()
    A = Projector(L, shape, [0.0, 0.0, 0.0], size, tof=(3.66, 649.2))
    x = torch.rand((5,) + shape, device="cuda", requires_grad=True)
    y = torch.rand((5, 20000), device="cuda")
    (A(x) * y).sum().backward()
    for b in range(5):
        xb = x[b].detach().clone().requires_grad_(True)
        p = A(xb)
        (p * y[b]).sum().backward()
        assert torch.equal(p, A(x)[b]) and torch.equal(x.grad[b], xb.grad)
    xk = x.detach().permute(0, 3, 2, 1).contiguous()
    want = A.plan.project_batch(xk)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = A.plan.project_batch(xk)
    for _ in range(2):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)


def test_refused():
    plan, n = _plan((16, 16, 8), (4.0, 4.0, 4.0), 100, False)
    from srf_amd import ops
    with pytest.raises(ValueError):
        plan.project_batch(torch.zeros((2, 8, 16, 15), device="cuda"))
    with pytest.raises(ValueError):
        ops.plan_backproject_batch(plan.handle, torch.zeros((2, n + 1), device="cuda"), n, plan.shape, 1)
    with pytest.raises(ValueError):
        plan.project_batch(torch.zeros((2, 8, 16, 16)))
    assert plan.project_batch(torch.zeros((0, 8, 16, 16), device="cuda")).shape == (0, n)
