"""One-shot backprojection of a long list: every voxel as exact as the float atomics of the
same events in short lists, whatever the range of the terms.

Both evaluate a term by the same float operations, so that the two differ by the rounding
of the sums alone: 500 half-ulps as in test_gpu_binned.py, relative to the voxel itself,
and below float32's normal range (2^-126 a term) nothing is compared."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

REL, TINY = 500 * 2.0 ** -24, 5000 * 2.0 ** -126
SHAPE, VOXEL, N, STEP = (128, 128, 17), (4.0, 4.0, 4.0), 45000, 5000
GEOM = [0.0, 0.0, 0.0] + [a * b for a, b in zip(SHAPE, VOXEL)]


def _lors(seed, tof_sigma=10.0):
    """Lines across the whole image whose TOF centres lie within a few cm of the axis."""
    rng = np.random.default_rng(seed)
    phi = rng.uniform(0, 2 * np.pi, N)
    psi = phi + np.pi + rng.normal(0, 0.5, N)
    z = rng.uniform(-30, 30, (N, 2))
    L = np.stack([400 * np.cos(phi), 400 * np.sin(phi), z[:, 0], 400 * np.cos(psi), 400 * np.sin(psi), z[:, 1],
                  rng.normal(0, tof_sigma, N)], 1)
    return torch.from_numpy(L.astype(np.float32)).cuda()


def _both(L, v, mode, tof=True):
    from srf_amd import ops
    args = (list(SHAPE), GEOM, tof, 3.66, 649.2, mode)
    long = ops.backproject(L, v, *args)
    short = sum(ops.backproject(L[k:k + STEP].contiguous(), v[k:k + STEP].contiguous(), *args).double()
                for k in range(0, N, STEP))
    return long.double(), short


def _check(long, short):
    fin = torch.isfinite(short)
    assert torch.equal(torch.isnan(long), torch.isnan(short)) and torch.equal(torch.isinf(long), torch.isinf(short))
    err = (long - short).abs()[fin]
    bound = REL * short.abs()[fin] + TINY
    print("worst", float((err / bound).max()), "smallest voxel", float(short[fin & (short > 0)].min()), flush=True)
    assert bool((err <= bound).all())


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("seed", [1, 2])
def test_tails_of_the_tof_gaussian(mode, seed):
    L = _lors(seed)
    v = torch.rand(N, generator=torch.Generator(device="cuda").manual_seed(seed), device="cuda") + 0.1
    long, short = _both(L, v, mode)
    assert float(short.min()) < 1e-12 * float(short.max())   # the tails are there
    _check(long, short)


@pytest.mark.parametrize("tof", [False, True])
@pytest.mark.parametrize("mode", [0, 1])
def test_wide_values_and_lengths(tof, mode):
    """Values over 60 binary orders of magnitude, lines of 50 to 800 mm."""
    L = _lors(5, 60.0)
    g = torch.Generator(device="cuda").manual_seed(7)
    v = torch.exp2(60 * torch.rand(N, generator=g, device="cuda") - 30)
    short_lines = torch.arange(N, device="cuda") % 3 == 0
    mid, half = 0.5 * (L[:, :3] + L[:, 3:6]), 0.5 * (L[:, 3:6] - L[:, :3])
    L[short_lines, :3] = (mid - half * 0.0625)[short_lines]
    L[short_lines, 3:6] = (mid + half * 0.0625)[short_lines]
    _check(*_both(L if tof else L[:, :6].contiguous(), v, mode, tof))


@pytest.mark.parametrize("mode", [0, 1])
def test_values_that_are_not_finite(mode):
    """NaN and infinite values, and a TOF value that is not a number, reach the voxels that
    their events touch and no others."""
    L = _lors(9)
    v = torch.rand(N, device="cuda") + 0.1
    v[100], v[20000], v[20001] = float("nan"), float("inf"), 0.0
    L[31000, 6] = float("nan")
    L[32000, 6] = float("inf")
    _check(*_both(L, v, mode))
