"""The GPU Delaunay where its work is dealt out: point counts around the runs
that the XCDs take in turn (512 points: 8 XCDs x 64), and spheres whose grid
columns hold a dense cluster (their points shared by a wavefront)."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _points(kind, n):
    rng = np.random.default_rng(n)
    if kind == "uniform":
        return rng.random((n, 3)).astype(np.float32)
    # a dense cluster inside a sparse shell: a hull tetrahedron's sphere is as
    # wide as the scene, and a coarse cell holds most of the points
    k = n * 9 // 10
    d = rng.normal(size=(n - k, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    return np.concatenate([0.02 * rng.normal(size=(k, 3)) + [0.3, -0.2, 0.1],
                           d * rng.uniform(4.0, 16.0, (n - k, 1))]).astype(np.float32)


@pytest.mark.parametrize("kind", ["uniform", "cluster"])
@pytest.mark.parametrize("n", [32, 63, 65, 511, 512, 513, 1025, 20_011])
def test_same_tetrahedra_as_qhull(kind, n):
    """Whole numbers: every table equals Qhull's, after a rebuild and after an
    incremental one."""
    import torch

    import sdfoam_amd

    print(f"delaunay runs {kind} n={n}", flush=True)
    raw = torch.from_numpy(_points(kind, n)).cuda()
    tri = sdfoam_amd.Triangulation(raw)
    p = raw[tri.permutation().view(torch.int32).long()].contiguous()
    rng = np.random.default_rng(n + 1)
    _, radius = sdfoam_amd.farthest_neighbor(p, tri.point_adjacency(),
                                             tri.point_adjacency_offsets())
    step = torch.from_numpy(rng.normal(size=(n, 3)).astype(np.float32)).cuda()
    for pts in (p, p + 1e-3 * radius[:, None] * step):
        if pts is not p:
            tri.rebuild(pts, incremental=True)
        ref = sdfoam_amd.Triangulation(pts, method="qhull")
        # the reference sorts its points again: map its ids back
        perm = ref.permutation().view(torch.int32).long()
        want = perm[ref.tets().view(torch.int32).long()].sort(dim=1)[0]
        got = tri.tets().view(torch.int32).long().sort(dim=1)[0]
        assert torch.equal(torch.unique(got, dim=0), torch.unique(want, dim=0))
        assert got.shape == want.shape
        offs = tri.point_adjacency_offsets().view(torch.int32).long()
        edges = torch.unique(torch.cat([want[:, [i, j]] for i in range(4) for j in range(4)
                                        if i != j]), dim=0)
        assert torch.equal(tri.point_adjacency().view(torch.int32).long(), edges[:, 1])
        assert torch.equal(offs[1:] - offs[:-1], torch.bincount(edges[:, 0], minlength=n))
