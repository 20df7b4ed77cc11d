"""The forward and the backward with several lanes per ray, at the edges of the
rules that choose their number and of the tiles of 64 rays that share a row of
the walk record: every output of the forward and the record itself equal the
one-lane forward's (cell_table=False) bit for bit, and the backward meets the
oracle's bounds."""

import numpy as np
import pytest

from conftest import scene
from test_gpu_parity import (_backward_both, _check_backward, gamma, gpu_scene,  # noqa: F401
                             record_rows, torch_dev)

pytestmark = pytest.mark.gpu


def cut(w, shape):
    """The workload over `shape` rays ([R] or [H, W]) taken from its own, repeated."""
    import dataclasses

    n = int(np.prod(shape))
    i = np.arange(n) * 7 % w.num_rays

    def take(x, last):
        return np.ascontiguousarray(x.reshape(w.num_rays, -1)[i].reshape(tuple(shape) + (last,)))

    return dataclasses.replace(
        w, rays=take(w.rays, 6), quantiles=take(w.quantiles, 1), grad_rgba=take(w.grad_rgba, 4),
        depth_grad=take(w.depth_grad, 1),
        extra=dict(w.extra, start=w.extra["start"].reshape(-1)[i].reshape(tuple(shape))))


# C1 has 4,104 points, C2 100,000: 16, 8, 4 and 2 lanes per ray and one, on both
# sides of each line; images with sides off the 8- and 16-pixel tiles
SHAPES = [
    (1, (1,)), (1, (63,)), (1, (65,)), (1, (8193,)), (1, (7, 9)), (1, (65, 113)), (1, (91, 91)),
    (1, (257, 256)), (1, (163_841,)), (1, (66_000,)),
    (2, (16_385,)), (2, (201, 203)), (2, (49_153,)), (2, (203, 301)), (2, (401, 499)),
]


@pytest.mark.parametrize("mode", ["sdfoam", "standard"])
@pytest.mark.parametrize("cfg,shape", SHAPES)
def test_split_forward_same_bits(torch_dev, monkeypatch, cfg, shape, mode):
    import torch

    import sdfoam_amd
    from sdfoam_amd import pipeline

    allocate = pipeline.TracePlan.allocate_record

    def allocate_zeroed(self, budget, chunks=0):
        allocate(self, budget, chunks)
        self.entries.zero_()

    monkeypatch.setattr(pipeline.TracePlan, "allocate_record", allocate_zeroed)
    w = cut(scene(cfg, mode=mode), shape)
    g = gpu_scene(w, torch_dev)
    pipe = sdfoam_amd.create_pipeline(w.sh_degree)
    q = torch.from_numpy(w.quantiles).to(torch_dev)
    inv_t = torch.tensor([w.inv_s], device=torch_dev)
    # a budget that ends inside a chunk and inside the longer walks
    a, b = [pipe.trace_forward(**g, depth_quantiles=q, return_contribution=True, alpha_mode=mode,
                               inv_s=inv_t, record_walk=True, walk_budget=45, cell_table=ct)
            for ct in (False, True)]
    free = pipe.trace_forward(**g, depth_quantiles=q, alpha_mode=mode, inv_s=inv_t,
                              record_walk=False)
    torch.cuda.synchronize()

    def bits(t):
        return t.contiguous().view(torch.uint8).cpu().numpy()

    for k in ("rgba", "depth", "depth_indices", "num_intersections"):
        assert np.array_equal(bits(a[k]), bits(b[k])), k
        assert np.array_equal(bits(a[k]), bits(free[k])), k
    for x, y in zip(record_rows(a["trace_plan"]), record_rows(b["trace_plan"])):
        assert np.array_equal(np.asarray(x).view(np.uint8), np.asarray(y).view(np.uint8))
    ca, cb = (o["contribution"].double().cpu().numpy().ravel() for o in (a, b))
    # the same fp32 weights in two orders, one per ray and point at most
    assert (np.abs(ca - cb) <= 2 * gamma(w.num_rays) * np.abs(ca) + 1e-30).all()


@pytest.mark.parametrize("mode", ["sdfoam", "standard"])
@pytest.mark.parametrize("cfg,shape", [
    (1, (1,)), (1, (65,)), (1, (8193,)), (1, (65, 113)), (1, (90, 455)), (1, (41_000,)),
    (1, (70_000,)), (2, (16_385,)), (2, (203, 243)), (2, (301, 305)),
])
def test_split_backward(torch_dev, oracle_lib, cfg, shape, mode):
    w = cut(scene(cfg, mode=mode), shape)
    bwd, st, ref = _backward_both(w, torch_dev, oracle_lib, mode, ray_error=True, walk=True)
    _check_backward(bwd, st, ref, w)
    bwd, st, ref = _backward_both(w, torch_dev, oracle_lib, mode)  # scanning
    _check_backward(bwd, st, ref, w)


# one pixel (the caller's arrays), then 16, 4, 2 lanes and one over C1, 8 and 4 over C2
@pytest.mark.parametrize("mode,dtype", [("sdfoam", "float32"), ("standard", "float16")])
@pytest.mark.parametrize("cfg,width,height", [
    (1, 1, 1), (1, 9, 7), (1, 64, 64), (1, 91, 91), (1, 257, 255), (1, 300, 301), (1, 500, 501),
    (2, 131, 127), (2, 300, 301),
])
def test_split_render_same_image(torch_dev, cfg, width, height, mode, dtype):
    """The render over the frame's tables equals the one over the caller's
    arrays (sdf_trace_benchmark), pixel for pixel."""
    import ctypes as C

    import torch

    import sdfoam_amd
    from sdfoam_amd import _lib, scenes

    w = scene(cfg, mode=mode)
    g = gpu_scene(w, torch_dev)
    g["attributes"] = g["attributes"].to(getattr(torch, dtype))
    scene_args = [g[k] for k in ("points", "attributes", "point_adjacency",
                                 "point_adjacency_offsets")]
    diff = sdfoam_amd.prefetch_adjacent_diff(*(scene_args[i] for i in (0, 2, 3)))
    diff = diff[: scene_args[2].numel()].clone()
    diff[:, 3] = 7.0  # the fourth column is the caller's: not read
    pipe = sdfoam_amd.create_pipeline(w.sh_degree, dtype)
    cam = scenes.camera_dict(w.extra["camera"], width=width, height=height)
    start = g["start_point"].view(torch.int32).reshape(-1)[:1].clone().view(torch.uint32)
    inv = torch.tensor([w.inv_s], device=torch_dev)
    got = torch.zeros((height, width), dtype=torch.int32, device=torch_dev).view(torch.uint32)
    pipe.trace_benchmark(*scene_args, diff, cam, start, got, weight_threshold=1e-3,
                         alpha_mode=mode, inv_s=inv)
    want = torch.zeros_like(got.view(torch.int32))
    c = _lib.Camera()
    for key in ("position", "forward", "up", "right"):
        getattr(c, key)[:] = [float(x) for x in cam[key]]
    c.fov, c.width, c.height, c.model = cam["fov"], width, height, _lib.SDF_CAMERA_PINHOLE
    vis = _lib.Visualization()
    vis.bg_color[:] = [1.0, 1.0, 1.0]
    settings = pipe._settings(1e-3, None, mode, None)
    p = [t.data_ptr() for t in scene_args]
    _lib.check(_lib.lib().sdf_trace_benchmark(
        w.sh_degree, C.byref(settings), w.num_points, p[0], p[1], scene_args[2].numel(), p[2], p[3],
        diff.data_ptr(), diff.shape[0], C.byref(c), C.byref(vis), start.data_ptr(),
        want.data_ptr(), inv.data_ptr(), _lib.stream_handle(torch_dev)))
    assert torch.equal(got.view(torch.int32), want)
    assert len(torch.unique(want)) > 1 or width == 1
