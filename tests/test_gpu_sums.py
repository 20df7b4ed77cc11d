"""The backward's sums over many rays: how exactly they are added up, and the two
contracts of the C interface for the per-point outputs (added to, or written),
over every SH degree and both attribute types, against the oracle."""

import ctypes as C

import numpy as np
import pytest

from conftest import scene
from test_gpu_fp16 import assert_close_h, half_scene
from test_gpu_parity import U, assert_close_model, gpu_scene, sum_depth, to_dev, _threads

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_dev():
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda:0")


# ---- equal rays: every ray adds the same terms --------------------------------

# over 4,104 points 8,192 rays take 16 lanes each, up to 40,960 four and 65,536 two
@pytest.mark.parametrize("mode", ["sdfoam", "standard"])
@pytest.mark.parametrize("shape", [(64, 128), (64, 160), (256, 160), (256, 256), (8192,), (32768,)])
def test_equal_rays(torch_dev, shape, mode):
    """One ray many times.  The sharpness' gradient, the point errors and the start
    cell's row are sums of equal terms: the count times what a single ray gives.
    They are held in fp64 past a wavefront's own sum of at most 64 fp32 terms; in fp32,
    the running sum of thousands of equal terms rounds the same way for long."""
    import torch

    import sdfoam_amd

    w = scene(1, mode=mode)
    n = int(np.prod(shape))
    g1 = gpu_scene(w, torch_dev)
    r = w.num_rays // 2 + 32  # one ray through the middle
    start1 = g1.pop("start_point").view(torch.int32).reshape(-1)[r]
    ray1 = g1.pop("rays").reshape(-1, 6)[r]
    pipe = sdfoam_amd.create_pipeline(w.sh_degree)
    inv = torch.tensor([w.inv_s], device=torch_dev)

    def run(lead):
        def many(x):
            return x.expand(lead + tuple(x.shape)).contiguous()

        start = many(start1).view(torch.uint32)
        rays = many(ray1)
        out = pipe.trace_forward(**g1, rays=rays, start_point=start, alpha_mode=mode, inv_s=inv,
                                 record_walk=True)
        grad = many(torch.tensor([0.3, -0.7, 0.9, 0.4], device=torch_dev))
        return pipe.trace_backward(**g1, rays=rays, start_point=start, rgb_out=out["rgba"],
                                   grad_in=grad, ray_error=many(torch.tensor(0.7, device=torch_dev)),
                                   alpha_mode=mode, inv_s=inv)

    one, many = run((1,) * len(shape)), run(shape)

    def close(a, b):
        a, b = a.double().reshape(-1).cpu().numpy(), b.double().reshape(-1).cpu().numpy() * n
        # 64 additions in a wavefront, and the two results' own roundings
        assert (np.abs(a - b) <= 66 * U * np.abs(b)).all(), np.abs(a / np.where(b == 0, 1, b) - 1).max()

    s = int(start1)
    close(many["attr_grad"][s], one["attr_grad"][s])
    close(many["points_grad"][s], one["points_grad"][s])
    close(many["point_error"], one["point_error"])
    if mode == "sdfoam":
        # a wavefront's own sum of 64 / G equal terms is exact, and so are the rest
        want = np.float32(n * float(one["sharpness_grad"]))
        assert np.float32(float(many["sharpness_grad"])) == want != 0.0


# ---- the C interface's two contracts -------------------------------------------


def c_scene(w, dev, dtype):
    """The workload and one more point that no ray reaches (an odd number of
    points: fp16 outputs end inside a 4-byte word)."""
    import torch

    g = gpu_scene(w, dev)
    pts = torch.cat([g["points"], torch.full((1, 3), 50.0, device=dev)])
    attrs = torch.cat([g["attributes"], torch.ones((1, g["attributes"].shape[1]), device=dev)])
    offs = g["point_adjacency_offsets"].view(torch.int32)
    offs = torch.cat([offs, offs[-1:]])
    return (pts, attrs.to(dtype), g["point_adjacency"].view(torch.int32), offs, g["rays"],
            g["start_point"].view(torch.int32))


def buffer(n, dtype, dev, value):
    """n values and one more (fp16 atomics work on 4-byte words)."""
    import torch

    return torch.full((n + 1,), value, dtype=dtype, device=dev)


def trace(w, dev, dtype, mode, outputs, extra, value):
    """Forward and backward through the C interface, the per-point outputs
    holding `value` before.  extra: what lies behind the accumulator's rows."""
    import torch

    import sdfoam_amd
    from sdfoam_amd import _lib

    L = _lib.lib()
    half = dtype == torch.float16
    pts, attrs, adj, offs, rays, start = c_scene(w, dev, dtype)
    n, e, R, D = pts.shape[0], adj.numel(), w.num_rays, attrs.shape[1]
    q = to_dev(w.quantiles, dev)
    Q = q.shape[-1]
    settings = sdfoam_amd.create_pipeline(w.sh_degree, dtype)._settings(None, None, mode, None, rays)
    inv = torch.tensor([w.inv_s], device=dev)
    nb = int(L.sdf_trace_scratch_bytes(n, e))
    scratch = torch.empty(nb, dtype=torch.uint8, device=dev)

    def aligned(nbytes):
        t = torch.full((nbytes + 256,), 0xC1, dtype=torch.uint8, device=dev)
        return t, (t.data_ptr() + 255) & ~255

    out = {"contribution": buffer(n, dtype, dev, value), "alpha": buffer(n, torch.float32, dev, value)}
    rgba = torch.empty((R, 4), dtype=dtype, device=dev)
    depth = torch.empty((R, Q), device=dev)
    didx = torch.empty((R, Q), dtype=torch.int32, device=dev)
    nis = torch.empty(R, dtype=torch.int32, device=dev)
    p = [t.data_ptr() for t in (pts, attrs, adj, offs, rays, start)]
    cb = int(L.sdf_cell_table_bytes(w.sh_degree, int(half), n))
    cells, cells_ptr = aligned(cb)
    plan = _lib.TracePlanDesc()
    plan.cell_table, plan.cell_table_bytes, plan.outputs = cells_ptr, cb, outputs & 1
    stream = _lib.stream_handle(dev)
    _lib.check(L.sdf_trace_forward_planned(
        C.byref(plan), w.sh_degree, C.byref(settings), n, p[0], p[1], e, p[2], p[3], R, p[4], p[5],
        Q, q.data_ptr(), rgba.data_ptr(), depth.data_ptr(), didx.data_ptr(), nis.data_ptr(),
        out["contribution"].data_ptr(), inv.data_ptr(), out["alpha"].data_ptr(), scratch.data_ptr(),
        nb, stream))
    rows = int(L.sdf_grad_accum_bytes(w.sh_degree, n))
    ab = rows + {"rows": 0, "errors": (8 * n + 15) // 16 * 16,
                 "sums": int(L.sdf_grad_sums_bytes(w.sh_degree, n))}[extra]
    accum, accum_ptr = aligned(ab)
    plan = _lib.TracePlanDesc()
    plan.grad_accum, plan.grad_accum_bytes, plan.outputs = accum_ptr, ab, outputs
    for k, m, dt in (("points_grad", 3 * n, torch.float32), ("attr_grad", D * n, dtype),
                     ("point_error", n, dtype), ("sharpness_grad", 1, torch.float32)):
        out[k] = buffer(m, dt, dev, value)
    g = to_dev(w.grad_rgba, dev).to(dtype)
    dg = to_dev(w.depth_grad, dev)
    err = to_dev(np.random.default_rng(11).uniform(0, 1, R).astype(np.float32), dev).to(dtype)
    _lib.check(L.sdf_trace_backward_planned(
        C.byref(plan), w.sh_degree, C.byref(settings), n, p[0], p[1], e, p[2], p[3], R, p[4], p[5],
        Q, q.data_ptr(), didx.data_ptr(), rgba.data_ptr(), g.data_ptr(), dg.data_ptr(),
        err.data_ptr(), out["points_grad"].data_ptr(), out["attr_grad"].data_ptr(),
        out["point_error"].data_ptr(), inv.data_ptr(), out["sharpness_grad"].data_ptr(),
        scratch.data_ptr(), nb, stream))
    torch.cuda.synchronize()
    # nothing past the accumulator's end was written
    end = accum_ptr - accum.data_ptr() + ab
    assert (accum[end:] == 0xC1).all()
    for k, t in out.items():
        assert not t[-1].isfinite() if value != value else t[-1] == value, k
    res = {k: t[:-1].float().cpu().numpy() for k, t in out.items()}
    given = {"rgba": rgba.float().cpu().numpy(), "didx": didx.cpu().numpy().view(np.uint32),
             "grad": g.float().cpu().numpy(), "err": err.float().cpu().numpy()}
    return res, given, n, D


def check(w, res, given, n, D, mode, half, base, oracle_lib):
    """res == base + the oracle's gradients, base being exact in both types."""
    N = w.num_points
    rgba = given["rgba"].reshape(w.rays.shape[:-1] + (4,))
    ref = oracle_lib.trace_backward(
        w.sh_degree, w.points, w.attributes, w.adjacency, w.offsets, w.rays, w.extra["start"], rgba,
        given["grad"].reshape(rgba.shape), w.quantiles,
        given["didx"].reshape(w.quantiles.shape), w.depth_grad,
        given["err"].reshape(w.rays.shape[:-1]), alpha_mode=mode, inv_s=w.inv_s, threads=_threads())
    fwd = oracle_lib.trace_forward(
        w.sh_degree, w.points, w.attributes, w.adjacency, w.offsets, w.rays, w.extra["start"],
        w.quantiles, alpha_mode=mode, inv_s=w.inv_s, threads=_threads())
    R = w.num_rays

    def one(name, got, want, absolute, k):
        got = got.reshape(n, -1)
        want, absolute = want.reshape(N, -1), absolute.reshape(N, -1)
        k = np.broadcast_to(np.asarray(k), want.shape) if np.ndim(k) == 0 else np.reshape(k, want.shape)
        # the added base is one more term of the sum
        assert_close = assert_close_h if half and name != "points_grad" else assert_close_model
        assert_close(name, got[:N], want + base, absolute + abs(base), k + 1)
        assert (got[N:] == base).all(), f"{name}: the cell that no ray reaches"

    one("points_grad", res["points_grad"], ref.points_grad, ref.points_grad_abs, ref.points_grad_k)
    one("attr_grad", res["attr_grad"], ref.attr_grad, ref.attr_grad_abs, ref.attr_grad_k)
    one("point_error", res["point_error"], ref.point_error, np.abs(ref.point_error), R)
    one("contribution", res["contribution"], fwd.contribution, np.abs(fwd.contribution), R)
    assert_close_model("sharpness_grad", res["sharpness_grad"], np.array([ref.sharpness_grad + base]),
                       np.array([ref.sharpness_abs + abs(base)]),
                       np.array([min(ref.sharpness_k, sum_depth(w, ref)) + 1]))
    # alpha: one visiting ray's value where a ray visits, else as before
    visited = fwd.contribution.reshape(-1) != 0
    a = res["alpha"]
    assert np.isfinite(a).all() and (a[N:] == base).all()
    if base == 0.0:
        assert ((a >= 0) & (a <= 1)).all() and (a[:N][visited] != 0).any()


@pytest.mark.parametrize("dtype", ["float32", "float16"])
@pytest.mark.parametrize("degree,mode", [(0, "sdfoam"), (1, "standard"), (2, "sdfoam"),
                                         (3, "standard"), (3, "sdfoam")])
@pytest.mark.parametrize("extra", ["rows", "errors", "sums"])
def test_outputs_added_to(torch_dev, oracle_lib, degree, mode, dtype, extra):
    """outputs == 0: what the caller's outputs held stays in them."""
    import torch

    half = dtype == "float16"
    w = half_scene(1, mode, sh_degree=degree) if half else scene(1, mode=mode, sh_degree=degree)
    base = 0.5
    res, given, n, D = trace(w, torch_dev, getattr(torch, dtype), mode, 0, extra, base)
    check(w, res, given, n, D, mode, half, base, oracle_lib)


@pytest.mark.parametrize("dtype", ["float32", "float16"])
@pytest.mark.parametrize("degree,mode", [(0, "sdfoam"), (1, "standard"), (2, "sdfoam"),
                                         (3, "standard"), (3, "sdfoam")])
@pytest.mark.parametrize("outputs,extra", [(1, "rows"), (1, "errors"), (1, "sums"), (3, "sums")])
def test_outputs_written(torch_dev, oracle_lib, degree, mode, dtype, outputs, extra):
    """SDF_OUTPUTS_FRESH: every element is written, whatever was there (NaN)."""
    import torch

    half = dtype == "float16"
    w = half_scene(1, mode, sh_degree=degree) if half else scene(1, mode=mode, sh_degree=degree)
    res, given, n, D = trace(w, torch_dev, getattr(torch, dtype), mode, outputs, extra, float("nan"))
    check(w, res, given, n, D, mode, half, 0.0, oracle_lib)
