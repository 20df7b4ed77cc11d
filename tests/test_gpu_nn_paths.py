"""nn's ways with scratch (a scan of every point, the search over the tree, a
search over points sorted for the call) at the edges of their groups, against the host's exact nearest neighbour; queries with infinities and
NaN against the tree search."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_dev():
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda:0")


def _threads():
    import os

    return min(16, os.cpu_count() or 1)


def _way(n, m):
    """The way the library takes, by the scratch it asks for."""
    from sdfoam_amd import _lib

    need = int(_lib.lib().sdf_nn_scratch_bytes(n, m))
    return "tree" if need == 0 else "scan" if need == -(-8 * m // 256) * 256 else "sorted"


# groups of 64 points: 4,096 is the most with one level of boxes, 262,144 with two
@pytest.mark.parametrize("n,m,way", [
    (32, 1, "tree"), (33, 257, "tree"), (2048, 300, "scan"), (2049, 256, "scan"),
    (300_001, 65, "scan"), (1500, 66_000, "sorted"), (4096, 33_025, "tree"),
    (4097, 33_017, "sorted"), (262_144, 769, "sorted"), (262_145, 901, "sorted"),
])
def test_nn_paths(torch_dev, oracle_lib, n, m, way):
    import torch

    import sdfoam_amd
    from sdfoam_amd import _lib, scenes

    assert _way(n, m) == way
    rng = np.random.default_rng(n + m)
    pts = rng.normal(size=(n, 3)).astype(np.float32)
    pts[n // 2] = pts[n // 3]  # a tie: the smaller index wins
    pts[: n // 4, 2] = 0.25  # a plane: boxes without extent
    pts = np.ascontiguousarray(pts[scenes.sort_points_order(pts)])
    qs = (pts[rng.integers(0, n, m)] + rng.normal(0, 0.05, (m, 3))).astype(np.float32)
    qs[::3] = pts[rng.integers(0, n, qs[::3].shape[0])]  # on points
    qs[-1] = 1e3
    p = torch.from_numpy(pts).to(torch_dev)
    tree = sdfoam_amd.build_aabb_tree(p)
    got = sdfoam_amd.nn(p, tree, torch.from_numpy(qs).to(torch_dev))
    want = oracle_lib.nn(pts, qs, threads=_threads())
    assert np.array_equal(got.view(torch.int32).cpu().numpy().astype(np.uint32), want)
    # infinite and NaN coordinates: as the search over the tree gives
    odd = qs.copy()
    k = np.arange(m)
    odd[k % 50 == 7, 1] = np.inf
    odd[k % 50 == 8, 0] = -np.inf
    odd[k % 50 == 9, 2] = np.nan
    q = torch.from_numpy(odd).to(torch_dev)
    got = sdfoam_amd.nn(p, tree, q)
    want = torch.empty(m, dtype=torch.int32, device=torch_dev)
    _lib.check(_lib.lib().sdf_nn(p.data_ptr(), tree.data_ptr(), q.data_ptr(), n, m,
                                 want.data_ptr(), _lib.stream_handle(torch_dev)))
    assert torch.equal(got.view(torch.int32), want)


@pytest.mark.parametrize("n", [2, 3, 33, 2047, 2048, 2049, 4097, (1 << 21) + 1])
def test_tree_levels(torch_dev, n):
    """The tree's levels at the edges of the eleven that one launch makes:
    every node is the union of its two children."""
    import torch

    import sdfoam_amd

    g = torch.Generator(device="cpu").manual_seed(n)
    p = torch.randn((n, 3), generator=g).to(torch_dev)
    tree = sdfoam_amd.build_aabb_tree(p)
    n2 = tree.shape[0]
    assert torch.equal(tree[-1], torch.zeros_like(tree[-1]))
    pad = torch.cat([p, p[-1:].expand(n2 - n, 3)]).view(n2 // 2, 2, 3)
    level = torch.stack([pad.amin(1), pad.amax(1)], dim=1)
    at = 0
    while True:
        w = level.shape[0]
        assert torch.equal(tree[at:at + w], level), w
        if w == 1:
            break
        at += w
        pair = level.view(w // 2, 2, 2, 3)
        level = torch.stack([pair[:, :, 0].amin(1), pair[:, :, 1].amax(1)], dim=1)
