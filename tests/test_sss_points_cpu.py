"""Points handed to SingleScatterSimulation.line_integrals: refused or converted before
any address of theirs reaches the library (no GPU needed: the library is replaced)."""
import contextlib

import pytest
import torch

from srf_amd import ops, sss


class _NoCall:
    def __getattr__(self, name):
        raise AssertionError(f"{name} was called")


@pytest.fixture
def sim(monkeypatch):
    s = object.__new__(sss.SingleScatterSimulation)
    s.dev = torch.device("cpu")
    s.det, s.nd = torch.zeros(5, 4), 5
    s.shape, s.geom = [4, 3, 2], [0.0, 0.0, 0.0, 8.0, 6.0, 4.0]
    s.plan, s.pts_xyz = None, torch.zeros(7, 3)
    monkeypatch.setattr(ops, "to_kernel_layout", lambda x: x.permute(2, 1, 0).contiguous())
    monkeypatch.setattr(ops, "lib", lambda: _NoCall())
    monkeypatch.setattr(sss, "lib", lambda: _NoCall())
    monkeypatch.setattr(torch.cuda, "device", lambda d: contextlib.nullcontext())
    # a stand-in for the GPU: det and image (and points, unless they are host points) pass
    # the device test, which on a machine without one no tensor does
    req = ops._req
    s.host_points = False

    def stand_in(t, name, dtype=torch.float32):
        if name == "points" and s.host_points:
            return req(t, name, dtype)
        if t.dtype != dtype or not t.is_contiguous():
            raise ValueError(f"{name}: {t.dtype}")

    monkeypatch.setattr(ops, "_req", stand_in)
    return s


def test_host_points_are_refused(sim):
    sim.host_points = True
    with pytest.raises(ValueError, match="GPU tensor"):
        sim.line_integrals(torch.zeros(4, 3, 2), torch.zeros(6, 4))


@pytest.mark.parametrize("pts", [torch.zeros(6, 4, dtype=torch.float64), torch.zeros(6, 3, dtype=torch.complex64),
                                 torch.zeros(6, 2), torch.zeros(6), torch.zeros(2, 6, 4)])
def test_types_and_shapes_are_refused(sim, pts):
    with pytest.raises(ValueError):
        sim.line_integrals(torch.zeros(4, 3, 2), pts)


def test_image_of_another_size_is_refused(sim):
    with pytest.raises(ValueError, match="voxels"):
        sim.line_integrals(torch.zeros(4, 3, 3), torch.zeros(6, 4))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16, torch.int32, torch.int64])
def test_lower_precisions_are_converted(sim, monkeypatch, dtype):
    seen = {}

    def stand_in(det, points, image_k, shape, geom):
        seen["points"] = points
        return torch.zeros(det.shape[0], points.shape[0])

    monkeypatch.setattr(ops, "point_integrals", stand_in)
    pts = torch.arange(24).reshape(4, 6).t().to(dtype)        # columns contiguous
    assert sim.line_integrals(torch.zeros(4, 3, 2), pts).shape == (5, 6)
    got = seen["points"]
    assert got.dtype == torch.float32 and got.is_contiguous() and torch.equal(got, pts.float())
