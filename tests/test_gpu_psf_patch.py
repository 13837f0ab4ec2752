"""The register-blocked 11 x 11 patch kernel of srf_psf_xy against float64, at the
edges of its strips (8 pixels along j, 1-4 strips per workgroup), slice chunks (64
or 128 per wavefront) and image borders, both directions, with and without the
ratio.  All values are positive, so 121 fused multiply-adds of float32 are within
121 half-ulps (relative), and the ratio adds one addition and one division."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _blur64(x, w, nx, ny, adjoint):
    x = x.double().reshape(nx, ny, -1)
    w = w.double().reshape(nx, ny, 121)
    out = torch.zeros_like(x)
    for o in range(121):
        a, b = o // 11 - 5, o % 11 - 5
        i0, i1, j0, j1 = max(0, -a), min(nx, nx - a), max(0, -b), min(ny, ny - b)
        if i0 >= i1 or j0 >= j1:
            continue
        wt = w[i0:i1, j0:j1, o, None]
        if adjoint:
            out[i0:i1, j0:j1] += wt * x[i0 + a:i1 + a, j0 + b:j1 + b]
        else:
            out[i0 + a:i1 + a, j0 + b:j1 + b] += wt * x[i0:i1, j0:j1]
    return out.reshape(nx * ny, -1)


@pytest.mark.parametrize("shape", [(1, 1, 1), (3, 4, 5), (5, 8, 64), (12, 18, 65), (13, 19, 128), (9, 33, 129),
                                   (7, 31, 192), (6, 40, 256), (11, 17, 257), (20, 23, 512)])
def test_patch_kernel_matches_float64(shape):
    from srf_amd import psf
    nx, ny, nz = shape
    g = torch.Generator(device="cuda").manual_seed(nx * 1000 + nz)
    x = torch.rand((nx * ny, nz), generator=g, device="cuda") + 0.1
    w = torch.rand((nx * ny, 121), generator=g, device="cuda")
    d = torch.rand((nx * ny, nz), generator=g, device="cuda") + 0.5
    # weights whose target or source lies outside the image are never used
    o = torch.arange(121, device="cuda")
    a, b = o // 11 - 5, o % 11 - 5
    i = torch.arange(nx * ny, device="cuda") // ny
    j = torch.arange(nx * ny, device="cuda") % ny
    ti, tj = i[:, None] + a[None], j[:, None] + b[None]
    w[(ti < 0) | (ti >= nx) | (tj < 0) | (tj >= ny)] = float("nan")
    h = 2.0 ** -24
    for adj in (0, 1):
        want = _blur64(x, torch.nan_to_num(w), nx, ny, adj)
        got = psf.psf_xy(x, w, nx, ny, adj).double()
        print(shape, adj, float(((got - want).abs() / want).max()), flush=True)
        assert bool(((got - want).abs() <= 122 * h * want).all())
        got = psf.psf_xy(x, w, nx, ny, adj, d=d, eps=1e-16).double()
        want = d.double() / (want + 1e-16)
        assert bool(((got - want).abs() <= 125 * h * want).all())
