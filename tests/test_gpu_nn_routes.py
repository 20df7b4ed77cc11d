"""nn's three ways at the lines between them and at the edges of the scan's blocks,
against the host's exact nearest neighbour and the search over the tree; that search
by itself; and nn in a captured graph."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_dev():
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda:0")


def way(n, m):
    """The way the library takes, by the scratch it asks for."""
    from sdfoam_amd import _lib

    need = int(_lib.lib().sdf_nn_scratch_bytes(n, m))
    return "tree" if need == 0 else "scan" if need == -(-8 * m // 256) * 256 else "sorted"


def positions(n, m, seed, spread=True):
    from sdfoam_amd import scenes

    rng = np.random.default_rng(seed)
    pts = rng.normal(size=(n, 3)).astype(np.float32)
    pts[n // 2] = pts[n // 3]  # a tie: the smaller index wins
    if spread:
        pts[: n // 4, 2] = 0.25
        pts = np.ascontiguousarray(pts[scenes.sort_points_order(pts)])
    qs = (pts[rng.integers(0, n, m)] + rng.normal(0, 0.05, (m, 3))).astype(np.float32)
    qs[::3] = pts[rng.integers(0, n, qs[::3].shape[0])]
    qs[-1] = 1e3
    return pts, qs


def tree_search(p, tree, q):
    import torch

    from sdfoam_amd import _lib

    out = torch.full((q.shape[0],), -1, dtype=torch.int32, device=q.device)
    _lib.check(_lib.lib().sdf_nn(p.data_ptr(), tree.data_ptr(), q.data_ptr(), p.shape[0], q.shape[0],
                                 out.data_ptr(), _lib.stream_handle(q.device)))
    return out


# blocks of the scan: 2,048 points; up to 8,192 one block for all; 1, 2 and 64 queries per block
@pytest.mark.parametrize("n,m,route", [
    (32, 5, "tree"), (64, 70_000, "tree"), (65, 1, "scan"), (65, 2048, "scan"), (65, 2049, "scan"),
    (2048, 65_536, "scan"), (2048, 65_537, "sorted"), (2049, 2048, "scan"), (2049, 2049, "tree"),
    (4096, 2048, "scan"), (4096, 2049, "tree"), (4097, 33_016, "scan"), (4097, 33_017, "sorted"),
    (8192, 2047, "scan"), (8192, 16_640, "scan"), (8192, 16_641, "sorted"), (8193, 409, "scan"),
    (8193, 410, "scan"), (100_001, 1598, "scan"), (100_001, 1599, "sorted"),
    (262_145, 767, "scan"), (262_145, 769, "sorted"), (1_048_577, 383, "scan"),
    (1_048_577, 385, "sorted"), (2_000_001, 201, "scan"), (2_000_001, 202, "sorted"),
])
def test_routes(torch_dev, oracle_lib, n, m, route):
    import torch

    import sdfoam_amd

    assert way(n, m) == route
    pts, qs = positions(n, m, n + m, spread=n < 1_000_000)
    p = torch.from_numpy(pts).to(torch_dev)
    tree = sdfoam_amd.build_aabb_tree(p)
    # memory that the scratch may be taken from
    torch.full((max(8 * m, 64) // 4 + 128,), -1, dtype=torch.int32, device=torch_dev)
    got = sdfoam_amd.nn(p, tree, torch.from_numpy(qs).to(torch_dev)).view(torch.int32)
    some = np.unique(np.linspace(0, m - 1, min(m, 3000)).astype(int))
    want = oracle_lib.nn(pts, qs[some], threads=8)
    assert np.array_equal(got.cpu().numpy()[some].astype(np.uint32), want)
    if n < 1_000_000:
        odd = qs.copy()
        k = np.arange(m)
        odd[k % 50 == 7, 1] = np.inf
        odd[k % 50 == 8, 0] = -np.inf
        odd[k % 50 == 9, 2] = np.nan
        q = torch.from_numpy(odd).to(torch_dev)
        assert torch.equal(sdfoam_amd.nn(p, tree, q).view(torch.int32), tree_search(p, tree, q))


def test_four_levels_of_boxes(torch_dev):
    """Past 64^4 points the sorted search has four levels of boxes."""
    import torch

    import sdfoam_amd

    n, m = 64 ** 4 + 1, 100
    assert way(n, m) == "sorted"
    g = torch.Generator(device=torch_dev).manual_seed(5)
    p = torch.randn((n, 3), generator=g, device=torch_dev)
    q = torch.randn((m, 3), generator=g, device=torch_dev)
    q[::4] = p[torch.randint(0, n, (m // 4,), generator=g, device=torch_dev)]
    got = sdfoam_amd.nn(p, sdfoam_amd.build_aabb_tree(p), q).view(torch.int32).long()
    for k in range(m):
        d = (p - q[k]).double().square().sum(1)
        # the fp32 distances differ from these by at most 3 roundings
        assert d[got[k]] <= d.min() * (1 + 1e-6)


@pytest.mark.parametrize("n", [32, 33, 64, 65, 129, 4096, 4097, 70_000, 300_000])
def test_tree_search(torch_dev, oracle_lib, n):
    """The search over the caller's tree (sdf_nn) at every shape it distinguishes: one
    group of points, boxes of depth 6 and 12 in LDS, boxes below them; points in the
    reference's order and in none."""
    import torch

    import sdfoam_amd

    for spread in (True, False):
        pts, qs = positions(n, 2003, n, spread)
        p = torch.from_numpy(pts).to(torch_dev)
        got = tree_search(p, sdfoam_amd.build_aabb_tree(p), torch.from_numpy(qs).to(torch_dev))
        want = oracle_lib.nn(pts, qs, threads=8)
        assert np.array_equal(got.cpu().numpy().astype(np.uint32), want)


@pytest.mark.parametrize("n,m,route", [(2048, 3000, "scan"), (20_000, 100, "scan"),
                                       (4096, 3000, "tree"), (20_000, 30_000, "sorted")])
def test_captured(torch_dev, n, m, route):
    """In a captured graph the sorted way's call searches the tree (the sorts would
    record memset nodes).  Every replay, over new queries, equals the eager result."""
    import torch

    import sdfoam_amd

    assert way(n, m) == route
    pts, _ = positions(n, m, 3)
    p = torch.from_numpy(pts).to(torch_dev)
    tree = sdfoam_amd.build_aabb_tree(p)
    q = torch.zeros((m, 3), device=torch_dev)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        sdfoam_amd.nn(p, tree, q)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = sdfoam_amd.nn(p, tree, q)
    g = torch.Generator(device=torch_dev).manual_seed(n)
    for _ in range(4):
        q.copy_(torch.randn((m, 3), generator=g, device=torch_dev))
        want = sdfoam_amd.nn(p, tree, q).view(torch.int32).clone()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got.view(torch.int32), want)
