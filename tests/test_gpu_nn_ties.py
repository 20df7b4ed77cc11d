"""nn where many points are as near as the nearest one: queries with an infinite
coordinate or so far out that all distances round to one value, points that
coincide by the thousands.  The smallest index is found, and such queries cost
about what others do (their ties are not looked through one by one)."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = 300_001


@pytest.fixture(scope="module")
def data():
    import torch

    import sdfoam_amd
    from sdfoam_amd import scenes

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    rng = np.random.default_rng(3)
    pts = rng.uniform(-1, 1, (N, 3)).astype(np.float32)
    pts[rng.permutation(N)[: N // 4]] = (0.25, -0.5, 0.125)  # one place, N / 4 points
    pts = np.ascontiguousarray(pts[scenes.sort_points_order(pts)])
    p = torch.from_numpy(pts).cuda()
    return pts, p, sdfoam_amd.build_aabb_tree(p)


def queries(kind, m, rng):
    q = rng.uniform(-1, 1, (m, 3)).astype(np.float32)
    at = rng.permutation(m)[: m // 100]
    if kind == "infinite":
        q[at, rng.integers(0, 3, at.size)] = np.where(rng.random(at.size) < 0.5, np.inf, -np.inf)
    elif kind == "far":
        q[at] = (rng.choice([-1.0, 1.0], (at.size, 3)) * 1e12).astype(np.float32)
    elif kind == "duplicates":
        q[at] = (0.25, -0.5, 0.125)
    return q


def search(which, p, tree, q):
    """nn (sorted points for this many queries), or the search over the tree."""
    import torch

    import sdfoam_amd
    from sdfoam_amd import _lib

    if which == "nn":
        return sdfoam_amd.nn(p, tree, q).view(torch.int32)
    out = torch.empty(q.shape[0], dtype=torch.int32, device=q.device)
    _lib.check(_lib.lib().sdf_nn(p.data_ptr(), tree.data_ptr(), q.data_ptr(), p.shape[0], q.shape[0],
                                 out.data_ptr(), _lib.stream_handle(q.device)))
    return out


@pytest.mark.parametrize("which", ["nn", "tree"])
@pytest.mark.parametrize("kind", ["infinite", "far", "duplicates"])
def test_ties(data, oracle_lib, which, kind):
    import torch

    pts, p, tree = data
    q = queries(kind, 20_000, np.random.default_rng(17))
    got = search(which, p, tree, torch.from_numpy(q).cuda()).cpu().numpy().astype(np.uint32)
    some = np.concatenate([np.flatnonzero((np.abs(q) > 2).any(1) | (q == (0.25, -0.5, 0.125)).all(1)),
                           np.arange(0, 20_000, 97)])
    want = oracle_lib.nn(pts, q[some], threads=8)
    assert np.array_equal(got[some], want)


@pytest.mark.parametrize("kind", ["infinite", "far", "duplicates"])
def test_ties_cost(data, kind):
    """100,000 queries of which 1% tie with thousands of points take at most five
    times as long as without (looking through the ties took 8 to 40 times)."""
    import torch

    _, p, tree = data

    def ms(k):
        q = torch.from_numpy(queries(k, 100_000, np.random.default_rng(5))).cuda()
        times = []
        for _ in range(4):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            search("nn", p, tree, q)
            b.record()
            torch.cuda.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)

    plain, ties = ms("plain"), ms(kind)
    print(f"{kind}: {ties:.3f} ms against {plain:.3f}")
    assert ties <= 5.0 * plain
