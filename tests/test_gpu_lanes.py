"""The fp16 forward over the cell table, at every number of lanes per ray and with
the half-batch face loads of sorted rays, against the one-lane forward over the
caller's arrays (cell_table=False): every per-ray output and the walk record bit for
bit, contributions within the bound of their roundings; and the backward of either
dtype where the number of its lanes changes, against the oracle."""

import numpy as np
import pytest

from conftest import scene
from test_gpu_fp16 import gamma_h, half_scene
from test_gpu_parity import _backward_both, _check_backward, gpu_scene, record_rows, torch_dev  # noqa: F401
from test_gpu_split import cut

pytestmark = pytest.mark.gpu

# C1 has 4,104 points, C2 100,000.  16, 8, 4, 2 lanes and one (images), then batches:
# 16 lanes unsorted, 4, 2 and 1 sorted; rays sorted from 32,768 on
SHAPES = [(1, (7, 9)), (1, (64, 128)), (2, (150, 151)), (1, (200, 201)), (2, (201, 203)),
          (1, (300, 301)), (1, (420, 421)), (2, (401, 499)), (1, (65,)), (1, (8193,)),
          (1, (32_768,)), (1, (33_001,)), (2, (49_153,)), (2, (98_305,)), (1, (170_000,))]


@pytest.mark.parametrize("contribution", [False, True])
@pytest.mark.parametrize("mode", ["sdfoam", "standard"])
@pytest.mark.parametrize("cfg,shape", SHAPES)
def test_fp16_forward_same_bits(torch_dev, monkeypatch, cfg, shape, mode, contribution):
    import torch

    import sdfoam_amd
    from sdfoam_amd import pipeline

    allocate = pipeline.TracePlan.allocate_record

    def allocate_zeroed(self, budget, chunks=0):
        allocate(self, budget, chunks)
        self.entries.zero_()

    monkeypatch.setattr(pipeline.TracePlan, "allocate_record", allocate_zeroed)
    w = cut(half_scene(cfg, mode), shape)
    g = gpu_scene(w, torch_dev)
    g["attributes"] = g["attributes"].to(torch.float16)
    pipe = sdfoam_amd.create_pipeline(w.sh_degree, "float16")
    q = torch.from_numpy(w.quantiles).to(torch_dev)
    inv = torch.tensor([w.inv_s], device=torch_dev)
    a, b = [pipe.trace_forward(**g, depth_quantiles=q, return_contribution=contribution,
                               alpha_mode=mode, inv_s=inv, record_walk=True, walk_budget=45,
                               cell_table=ct) for ct in (False, True)]
    torch.cuda.synchronize()

    def bits(t):
        return t.contiguous().view(torch.uint8).cpu().numpy()

    for k in ("rgba", "depth", "depth_indices", "num_intersections"):
        assert np.array_equal(bits(a[k]), bits(b[k])), k
    for x, y in zip(record_rows(a["trace_plan"]), record_rows(b["trace_plan"])):
        assert np.array_equal(np.asarray(x).view(np.uint8), np.asarray(y).view(np.uint8))
    if contribution:
        ca, cb = (o["contribution"].double().cpu().numpy().ravel() for o in (a, b))
        # the same weights in two orders, every fp16 addition rounded
        assert (np.abs(ca - cb) <= 2 * gamma_h(w.num_rays) * np.abs(ca) + 1e-5).all()


# one lane at a full chip (over 600,000 image rays, 81,920 and 163,840 otherwise); four and two
# lanes on both sides of their lines
@pytest.mark.parametrize("cfg,shape", [(1, (90, 911)), (1, (81_920,)), (1, (81_921,)),
                                       (1, (256, 257)), (2, (448, 440)), (2, (501, 1201))])
def test_backward_lines(torch_dev, oracle_lib, cfg, shape):
    w = cut(scene(cfg), shape)
    bwd, st, ref = _backward_both(w, torch_dev, oracle_lib, "sdfoam", ray_error=True, walk=True)
    _check_backward(bwd, st, ref, w)
