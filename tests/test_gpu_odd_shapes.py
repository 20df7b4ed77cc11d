"""Inputs of shapes that the checks admit beside [N, 3] and [N, D]."""

import numpy as np
import pytest

from conftest import scene
from test_gpu_parity import gpu_scene, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float32", "float16"])
@pytest.mark.parametrize("grad_accum", [True, False])
def test_attribute_rows_past_the_points(dtype, grad_accum):
    """Points [N, 2, 3] with attributes [2 N, D]: the first N rows are traced,
    and the gradients of the others are 0, whatever the memory held."""
    import torch

    import sdfoam_amd

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    dev = torch.device("cuda:0")
    w = scene(1)
    g = gpu_scene(w, dev)
    n, d = g["attributes"].shape
    g["attributes"] = g["attributes"].to(getattr(torch, dtype))
    pipe = sdfoam_amd.create_pipeline(w.sh_degree, dtype)
    inv = torch.tensor([w.inv_s], device=dev)
    grad = to_dev(w.grad_rgba, dev).to(g["attributes"].dtype)

    def run(g):
        out = pipe.trace_forward(**g, alpha_mode="sdfoam", inv_s=inv, record_walk=True)
        # memory of the sizes that the backward takes next
        torch.full((2 * n * d + 1,), float("nan"), device=dev, dtype=g["attributes"].dtype)
        torch.full((2 * n, d), float("nan"), device=dev, dtype=g["attributes"].dtype)
        return pipe.trace_backward(**g, rgb_out=out["rgba"], grad_in=grad, alpha_mode="sdfoam",
                                   inv_s=inv, grad_accum=grad_accum)

    want = run(g)
    offs = g["point_adjacency_offsets"].view(torch.int32)
    odd = dict(g, points=torch.cat([g["points"], torch.zeros_like(g["points"])]).view(n, 2, 3),
               attributes=torch.cat([g["attributes"], torch.ones_like(g["attributes"])]),
               point_adjacency_offsets=torch.cat([offs, offs[-1:].expand(n)]).view(torch.uint32))
    got = run(odd)
    assert got["attr_grad"].shape == (2 * n, d)
    assert (got["attr_grad"][n:] == 0).all()
    a, b = got["attr_grad"][:n].float(), want["attr_grad"].float()
    # the same terms in another order: fp16 atomics round each addition
    tol = 1e-4 if dtype == "float32" else 2e-2 if grad_accum else 0.1
    assert ((a - b).norm() <= tol * b.norm())
    assert got["points_grad"].isfinite().all()
