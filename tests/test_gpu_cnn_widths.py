"""The elementwise network kernels with 16-byte runs of channels and one value at a time:
row lengths, offsets and addresses that allow the first and that do not.  Every result is
one rounding of exact or same-order sums, so all are compared bit for bit."""
import numpy as np
import pytest
import torch

import cnn_oracle as co
from test_gpu_cnn import DEV, _L, _bf, _f, _s

pytestmark = pytest.mark.gpu

D, H, W = 4, 6, 10
V = D * H * W
WIDTHS = [(16, 16, 16, 0, 0), (8, 24, 32, 8, 0), (12, 20, 16, 4, 0), (5, 7, 9, 3, 0), (16, 16, 16, 0, 1)]


def _rows(rng, n, stride, shift, bf):
    """n rows of `stride` values that start `shift` values into an allocation, and their values."""
    a = rng.normal(size=n * stride + shift)
    t, r = _bf(a) if bf else (torch.from_numpy(a.astype(np.float32)).to(DEV), a.astype(np.float32))
    return t[shift:], r[shift:].reshape(n, stride)


def _out(n, stride, shift, dtype):
    return torch.full((n * stride + shift,), 1, dtype=dtype, device=DEV)[shift:]


@pytest.mark.parametrize("C,xs,ys,off,shift", WIDTHS)
def test_pool_and_upsample(C, xs, ys, off, shift):
    rng = np.random.default_rng(C)
    x, xr = _rows(rng, V, xs, shift, True)
    y = _out(V // 8, ys, shift, torch.int16)
    assert _L().srf_cnn_pool(x.data_ptr(), D, H, W, C, xs, y.data_ptr(), ys, _s()) == 0
    got = _f(y).reshape(-1, ys)
    np.testing.assert_array_equal(got[:, :C], co.bf16_round(co.pool(xr[:, :C].reshape(D, H, W, C))).reshape(-1, C))
    u = _out(V, ys, shift, torch.int16)
    assert _L().srf_cnn_upsample(x.data_ptr(), D // 2, H // 2, W // 2, C, xs, u.data_ptr(), ys, off, _s()) == 0
    want = co.upsample(xr[:V // 8, :C].reshape(D // 2, H // 2, W // 2, C)).reshape(V, C)
    got = u.cpu().numpy().reshape(V, ys)
    np.testing.assert_array_equal(_f(u).reshape(V, ys)[:, off:off + C], want)
    assert np.all(np.delete(got, range(off, off + C), 1) == 1)


@pytest.mark.parametrize("C,xs,ys,off,shift", WIDTHS)
def test_gradients_and_copies(C, xs, ys, off, shift):
    rng = np.random.default_rng(C + 1)
    g, gr = _rows(rng, V, ys, shift, False)
    d = _out(V // 8, xs, shift, torch.float32)
    assert _L().srf_cnn_upsample_bwd(g.data_ptr(), D // 2, H // 2, W // 2, C, ys, off, d.data_ptr(), xs, _s()) == 0
    k = gr[:, off:off + C].reshape(D // 2, 2, H // 2, 2, W // 2, 2, C)
    want = np.zeros((D // 2, H // 2, W // 2, C), np.float32)
    for i in range(8):
        want = want + k[:, i >> 2, :, (i >> 1) & 1, :, i & 1]
    np.testing.assert_array_equal(d.cpu().numpy().reshape(-1, xs)[:, :C], want.reshape(-1, C))
    p = _out(V, xs, shift, torch.float32)
    assert _L().srf_cnn_pool_bwd(g.data_ptr(), D, H, W, C, ys, p.data_ptr(), xs, _s()) == 0
    want = co.upsample(gr[:V // 8, :C].reshape(D // 2, H // 2, W // 2, C)).reshape(V, C) * np.float32(0.125)
    np.testing.assert_array_equal(p.cpu().numpy().reshape(V, xs)[:, :C], want)
    for bf, add in ((0, 0), (0, 1), (1, 0)):
        x, xr = _rows(rng, V, xs, shift, bool(bf))
        y, yr = _rows(rng, V, ys, shift, bool(bf))
        assert _L().srf_cnn_copy_channels(x.data_ptr(), V, C, xs, 0, y.data_ptr(), ys, off, 1 - bf, add, _s()) == 0
        want = yr.copy()
        want[:, off:off + C] = xr[:, :C] + (yr[:, off:off + C] if add else 0)
        np.testing.assert_array_equal((_f(y) if bf else y.cpu().numpy()).reshape(V, ys), want)


@pytest.mark.parametrize("C,das,as_,Cp,shift", [(16, 16, 16, 16, 0), (8, 12, 24, 16, 0), (1, 1, 1, 8, 0), (20, 21, 20, 24, 0),
                                                (16, 16, 16, 16, 1)])
@pytest.mark.parametrize("slope", [0.25, -1.0])
def test_activation_gradient(C, das, as_, Cp, shift, slope):
    rng = np.random.default_rng(Cp)
    g, gr = _rows(rng, V, das, shift, False)
    a, ar = _rows(rng, V, as_, shift, True)
    p = _out(V, Cp, shift, torch.int16)
    assert _L().srf_cnn_act_bwd(g.data_ptr(), das, a.data_ptr(), as_, V, C, Cp, slope, p.data_ptr(), _s()) == 0
    want = np.zeros((V, Cp))
    want[:, :C] = np.where((slope < 0) | (ar[:, :C] > 0), gr[:, :C], np.float32(slope) * gr[:, :C])
    np.testing.assert_array_equal(_f(p).reshape(V, Cp), co.bf16_round(want))
