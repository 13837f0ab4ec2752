"""The weight gradient (k_conv_wgrad_tr) at the edges of its 8 x 8 x 4 tiles and 16-channel
blocks, against the CPU float64 oracle.

Inputs are bf16 values, so every product is exact in float32 and only the sums round: an
element sums V products, so it may be off by V 2^-23 times the sum of their magnitudes
(one unit in the last place per addition)."""
import numpy as np
import pytest
import torch

import cnn_oracle as co
from test_gpu_cnn import DEV, _L, _bf, _s

pytestmark = pytest.mark.gpu


def _case(N, dims, cin_p, cout, taps, seed):
    from srf_amd.surrogate import _c8, _c32
    rng = np.random.default_rng(seed)
    x, xr = _bf(rng.normal(size=(N,) + dims + (cin_p,)))
    g = np.zeros((N,) + dims + (_c8(cout),))
    g[..., :cout] = rng.normal(size=(N,) + dims + (cout,))
    g, gr = _bf(g)
    gr = gr[..., :cout]
    want = sum(co.conv3d_grad_weight(xr[i], gr[i], taps) for i in range(N))
    size = sum(co.conv3d_grad_weight(abs(xr[i]), abs(gr[i]), taps) for i in range(N))
    V = N * int(np.prod(dims))
    dw = torch.zeros((taps, _c32(cout), cin_p), device=DEV)
    db = torch.zeros(cout, device=DEV)

    def run():
        assert _L().srf_cnn_conv_wgrad_batch(x.data_ptr(), g.data_ptr(), _c8(cout), N, *dims, cin_p, cout, _c32(cout),
                                             taps, dw.data_ptr(), db.data_ptr(), _s()) == 0

    def verify(times):
        got = dw.double().cpu().numpy()
        n = (V + times) * 2.0 ** -23
        assert np.all(abs(got[:, :cout] - times * want) <= times * n * size)
        assert np.all(got[:, cout:] == 0)
        flat = gr.reshape(-1, cout)
        assert np.all(abs(db.double().cpu().numpy() - times * flat.sum(0)) <= times * n * abs(flat).sum(0))

    return run, verify


@pytest.mark.parametrize("taps", [27, 1])
@pytest.mark.parametrize("N,dims,cin_p,cout", [
    (1, (1, 1, 1), 8, 1),            # one voxel
    (2, (3, 5, 12), 16, 16),         # ragged in every direction, two samples
    (1, (8, 16, 24), 8, 16),         # whole tiles, half a channel block
    (2, (5, 9, 8), 48, 16),          # dY shifted, three blocks of X
    (1, (4, 8, 17), 96, 32),         # dY shifted, two blocks of each
    (3, (4, 6, 16), 24, 40),         # part of a block on both sides
    (1, (4, 8, 8), 16, 72),          # X shifted, several blocks of dY
    (2, (4, 4, 8), 64, 64),
])
def test_weight_gradient_tiles(N, dims, cin_p, cout, taps):
    run, verify = _case(N, dims, cin_p, cout, taps, 3)
    run()
    verify(1)
    run()   # adds to what is there
    verify(2)


def test_weight_gradient_in_a_graph():
    """Under capture the sums are added without scratch."""
    run, verify = _case(2, (6, 16, 16), 48, 16, 27, 4)
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=side):
        run()
    graph.replay()
    torch.cuda.synchronize()
    verify(1)
    run()
    graph.replay()
    torch.cuda.synchronize()
    verify(3)
