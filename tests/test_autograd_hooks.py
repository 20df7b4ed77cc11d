"""Which backward TraceRays calls: the package's own one directly, and any
other trace_backward (a subclass', an instance's, one set on the class by a
profiler or a test) as it is."""

import types

import torch

from sdfoam_amd import render
from sdfoam_amd.pipeline import Pipeline

N, D, R = 5, 4, 3


def results(attr):
    return {"points_grad": torch.full((N, 3), float("nan")), "attr_grad": torch.full((N, D), attr),
            "sharpness_grad": torch.ones(1), "ray_grad": torch.zeros((R, 6))}


def backward(pipeline):
    """TraceRays.backward over a context as its forward leaves it."""
    ctx = types.SimpleNamespace(
        pipeline=pipeline, points=torch.zeros((N, 3)), attributes=torch.zeros((N, D)),
        point_adjacency=None, point_adjacency_offsets=None, rays=torch.zeros((R, 6)),
        start_point=None, rgba=torch.zeros((R, 4)), depth_quantiles=None, depth_indices=None,
        errbox=render.ErrorBox(), use_sdfoam=True, inv_s=torch.ones(1), eps=1e-6, sdf_channel=None)
    ctx.errbox.ray_error = None
    return render.TraceRays.backward(ctx, torch.ones((R, 4)), None, None, None, None, None)


def calls(monkeypatch):
    """The calls of Pipeline's own backward, which needs no GPU here."""
    seen = []

    def own(self, *args, **kw):
        seen.append(kw)
        return results(1.0)

    monkeypatch.setattr(Pipeline, "_backward", own)
    return seen


def test_own_backward(monkeypatch):
    seen = calls(monkeypatch)
    backward(Pipeline(0, torch.float32))
    assert len(seen) == 1 and seen[0]["autograd"] is True


def test_replaced_backwards_are_called(monkeypatch):
    """On the class, on a subclass and on an instance; what it returns is used
    (non-finite gradients as 0) and eps is handed on."""
    seen = calls(monkeypatch)
    given = []

    def hook(self, *args, **kw):
        given.append(kw)
        return results(2.0)

    class Sub(Pipeline):
        trace_backward = hook

    one = Pipeline(0, torch.float32)
    one.trace_backward = types.MethodType(hook, one)
    grads = [backward(Sub(0, torch.float32)), backward(one)]
    monkeypatch.setattr(Pipeline, "trace_backward", hook)
    grads.append(backward(Pipeline(0, torch.float32)))
    assert not seen and len(given) == 3
    for g, kw in zip(grads, given):
        assert kw["eps"] == 1e-6
        assert (g[1] == 0).all() and (g[2] == 2.0).all()


def test_class_wrapper_reaches_the_own_backward(monkeypatch):
    """A wrapper on the class that calls what it replaced (a profiler)."""
    seen = calls(monkeypatch)
    count = []
    inner = Pipeline.trace_backward

    def wrapper(self, *args, **kw):
        count.append(1)
        return inner(self, *args, **kw)

    monkeypatch.setattr(Pipeline, "trace_backward", wrapper)
    backward(Pipeline(0, torch.float32))
    assert len(count) == 1 and len(seen) == 1 and not seen[0].get("autograd")
