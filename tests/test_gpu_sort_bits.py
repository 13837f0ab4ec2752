"""Plans on both sides of the tile counts at which the record sort leaves its lowest key
bit out: every event's terms stay the same (digests, bit for bit), and backprojections
agree with short lists within the bounds of test_gpu_binned."""
import pytest
import torch

from test_gpu_binned import _close, _lors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("tiles", [1024, 1025, 2048, 2049])
def test_plan_at_tile_counts(tiles, mode):
    from srf_amd import ops
    n, shape = 20000, [30, 31, 8 * tiles - 3]
    geom = [0.3, -0.2, 0.5, 90.0, 93.0, 0.02 * shape[2]]
    L = _lors(n, tiles)
    v = torch.rand(n, generator=torch.Generator(device="cuda").manual_seed(4), device="cuda") + 0.1
    print("tiles", tiles, mode, flush=True)
    plan = ops.Plan(L, shape, geom, True, 3.66, 649.2)
    for a, b in zip(plan.digest(mode), ops.lor_digest(L, shape, geom, True, 3.66, 649.2, mode)):
        assert torch.equal(a, b)
    step = 4000
    want = sum(ops.backproject(L[k:k + step].contiguous(), v[k:k + step].contiguous(), shape, geom, True, 3.66, 649.2,
                               mode).double() for k in range(0, n, step))
    _close(plan.backproject(v, mode), want)
    plan.close()
