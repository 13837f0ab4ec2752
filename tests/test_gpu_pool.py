"""Scratch and plan memory from the block pool, on several streams and host threads."""
import threading

import pytest
import torch

from test_gpu_binned import _lors

pytestmark = pytest.mark.gpu


def test_streams_and_threads():
    """Long one-shot calls and plans of several host threads, each on a stream of its own, all
    through the pool: the results of the same calls one after the other."""
    from srf_amd import ops
    shape, geom = [64, 60, 17], [0.0, 0.0, 0.0, 128.0, 120.0, 34.0]
    lists = [_lors(90000 + 1000 * k, 20 + k)[8:].contiguous() for k in range(4)]
    img = torch.rand((17, 60, 64), device="cuda")
    big = torch.rand((90, 140, 150), device="cuda")   # above BUNDLE_IMAGE_MIN
    bshape, bgeom = [150, 140, 90], [0.0, 0.0, 0.0, 150.0, 140.0, 90.0]

    def work(L):
        bp = ops.backproject(L, None, shape, geom, True, 3.66, 649.2, 0)
        plan = ops.Plan(L, shape, geom, True, 3.66, 649.2)
        p, q = plan.project(img), plan.backproject(None, 0)
        plan.close()
        b = torch.cat([L, L]).contiguous()
        return bp, p, q, ops.project(b, big, bshape, bgeom, True, 3.66, 649.2)

    want = [work(L) for L in lists]
    torch.cuda.synchronize()
    out, errors = [None] * 4, []

    def run(k):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(5):
                    out[k] = work(lists[k])
                torch.cuda.current_stream().synchronize()
        except Exception as e:
            errors.append(e)

    ts = [threading.Thread(target=run, args=(k,)) for k in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errors, errors
    for got, ref in zip(out, want):
        assert torch.equal(got[1], ref[1]) and torch.equal(got[2], ref[2]) and torch.equal(got[3], ref[3])
        assert bool(((got[0] - ref[0]).abs() <= 2.0 ** -20 * ref[0]).all())   # float64 sums in any order


def test_block_goes_to_another_stream():
    """Scratch given back on one stream while its kernels run, taken on another at once."""
    from srf_amd import ops
    shape, geom = [150, 140, 90], [0.0, 0.0, 0.0, 150.0, 140.0, 90.0]
    img = torch.rand((90, 140, 150), device="cuda")
    L = _lors(400000, 31)[8:].contiguous()
    M = _lors(400000, 32)[8:].contiguous()
    a, b = (ops.project(x, img, shape, geom, True, 3.66, 649.2) for x in (L, M))
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(4)]
    outs = []
    for k in range(12):
        with torch.cuda.stream(streams[k % 4]):
            outs.append(ops.project(M if k % 2 else L, img, shape, geom, True, 3.66, 649.2))
    torch.cuda.synchronize()
    for k, o in enumerate(outs):
        assert torch.equal(o, b if k % 2 else a), k
