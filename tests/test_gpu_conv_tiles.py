"""The convolution kernels (k_conv, k_conv_rows, k_conv_res) at the edges of their tiles,
channel blocks and chunks, against the CPU float64 oracle.

Inputs and weights are bf16 values, so products are exact in float32 and an output is off
by at most one unit in the last place per addition: (27 cin + 2) 2^-23 of the sum of the
terms' magnitudes; a bf16 result adds its own rounding, 2^-8 of the value."""
import numpy as np
import pytest
import torch

import cnn_oracle as co
from test_gpu_cnn import DEV, _L, _bf, _f, _pad_w, _s

pytestmark = pytest.mark.gpu

BIG = (4, (7, 125, 125))       # k_conv_res: ragged in every direction, a sample per tile layer
MID = (2, (5, 61, 125))        # k_conv_rows
NARROW = (4, (24, 88, 24))     # k_conv, a slice per wavefront (24 columns are not 16s)
SOME = (1, (20, 64, 56))       # k_conv, two wavefronts a slice
FEW = (3, (3, 9, 17))          # k_conv, four


def _want(x, cc, w, b, slope):
    """Oracle and bound of the convolution of x's samples (cc > 0: of fine and coarse)."""
    if cc:
        f, c = x
        x = np.concatenate([c.repeat(2, 1).repeat(2, 2).repeat(2, 3), f], -1)
    y = np.stack([co.conv3d(v, w, b) for v in x])
    size = np.stack([co.conv3d(abs(v), abs(w), abs(b)) for v in x])
    return np.where(y < 0, slope * y, y) if slope >= 0 else y, size


@pytest.mark.parametrize("where,cin,cout,taps", [
    (BIG, 8, 16, 27), (BIG, 16, 16, 27), (BIG, 32, 9, 27), (BIG, 48, 16, 27), (BIG, 16, 48, 27),
    (MID, 24, 16, 27), (MID, 40, 32, 27), (MID, 16, 64, 27),
    (NARROW, 32, 20, 27), (NARROW, 8, 64, 27), (NARROW, 16, 1, 27),
    (SOME, 72, 16, 27), (FEW, 24, 40, 27), (FEW, 64, 64, 27), (NARROW, 40, 24, 1),
])
def test_convolution_tiles(where, cin, cout, taps):
    from srf_amd.surrogate import _c32
    N, dims = where
    rng = np.random.default_rng(cin + cout)
    x, xr = _bf(rng.normal(size=(N,) + dims + (cin,)))
    w, wr = _bf(_pad_w(rng.normal(size=(taps, cout, cin)), _c32(cout), cin))
    b = rng.normal(size=cout).astype(np.float32)
    want, size = _want(xr, 0, wr[:, :cout], b.astype(np.float64), 0.25)
    V, bd = N * int(np.prod(dims)), torch.from_numpy(b).to(DEV)
    bound = (taps * cin + 2) * 2.0 ** -23 * size
    for stride, off in ((cout, 0), (cout + 3, 2)):   # rows that vectors fit, and rows that they do not
        yf = torch.full((V, stride), 7.0, device=DEV)
        yb = torch.full((V, stride), 3, dtype=torch.int16, device=DEV)
        assert _L().srf_cnn_conv_batch(x.data_ptr(), w.data_ptr(), bd.data_ptr(), N, *dims, cin, cout, _c32(cout), taps,
                                       stride, off, 0.25, yb.data_ptr(), yf.data_ptr(), _s()) == 0
        torch.cuda.synchronize()
        cols = slice(off, off + cout)
        err = abs(yf[:, cols].double().cpu().numpy().reshape(want.shape) - want)
        assert np.all(err <= bound), err.max()
        err = abs(_f(yb[:, cols]).astype(np.float64).reshape(want.shape) - want)
        assert np.all(err <= bound + 2.0 ** -8 * abs(want))
        keep = [c for c in range(stride) if not off <= c < off + cout]
        assert bool((yf[:, keep] == 7.0).all()) and bool((yb[:, keep] == 3).all())


@pytest.mark.parametrize("where,cc,cf", [((4, (8, 126, 126)), 32, 16), ((2, (6, 62, 126)), 64, 32), ((2, (4, 6, 18)), 16, 8)])
def test_upsampled_input_tiles(where, cc, cf):
    from srf_amd.surrogate import _c32
    N, dims = where
    cout, cin = 16, cc + cf
    rng = np.random.default_rng(cc)
    f, fr = _bf(rng.normal(size=(N,) + dims + (cf,)))
    c, cr = _bf(rng.normal(size=(N,) + tuple(v // 2 for v in dims) + (cc,)))
    w, wr = _bf(_pad_w(rng.normal(size=(27, cout, cin)), _c32(cout), cin))
    y = torch.zeros((N * int(np.prod(dims)), cout), device=DEV)
    assert _L().srf_cnn_conv_up_batch(f.data_ptr(), c.data_ptr(), cc, w.data_ptr(), None, N, *dims, cin, cout,
                                      _c32(cout), 27, cout, 0, -1.0, None, y.data_ptr(), _s()) == 0
    torch.cuda.synchronize()
    want, size = _want((fr, cr), cc, wr[:, :cout], np.zeros(cout), -1.0)
    err = abs(y.double().cpu().numpy().reshape(want.shape) - want)
    assert np.all(err <= (27 * cin + 2) * 2.0 ** -23 * size)


@pytest.mark.parametrize("where,cin,cout", [(BIG, 16, 16), (MID, 24, 32), (SOME, 16, 16), (FEW, 16, 24), (FEW, 8, 64)])
def test_head_tiles(where, cin, cout):
    """The head sums the bf16 values that the layer stored."""
    from srf_amd.surrogate import _c32
    N, dims = where
    rng = np.random.default_rng(cout)
    x, _ = _bf(rng.normal(size=(N,) + dims + (cin,)))
    w, _ = _bf(_pad_w(rng.normal(size=(27, cout, cin)), _c32(cout), cin))
    hw, hr = _bf(rng.normal(size=cout))
    V, hb = N * int(np.prod(dims)), torch.tensor([0.5], device=DEV)
    y, out = torch.zeros((V, cout), dtype=torch.int16, device=DEV), torch.zeros(V, device=DEV)
    assert _L().srf_cnn_conv_head_batch(x.data_ptr(), w.data_ptr(), None, N, *dims, cin, cout, _c32(cout), 27, 0.01,
                                        y.data_ptr(), hw.data_ptr(), hb.data_ptr(), out.data_ptr(), _s()) == 0
    torch.cuda.synchronize()
    terms = _f(y).astype(np.float64) * hr
    err = abs(out.double().cpu().numpy() - (terms.sum(1) + 0.5))
    assert np.all(err <= (cout + 2) * 2.0 ** -23 * (abs(terms).sum(1) + 0.5))
