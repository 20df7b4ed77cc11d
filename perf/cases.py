"""What is measured: the work a program that trains or shows a Voronoi foam has this
package do, through the entry points it calls.

* train: a training step as a scene and its training loop run it: start cells of the
  rays' origins (``get_starting_point``), ``TraceRays`` and the gradients autograd
  asks of it.  Whole images (every ray of one camera, shaped [H, W, 6]) or batches of
  random rays of many cameras ([R, 6]), where the points have moved since the
  adjacency was built;
* eval: the same trace without gradients (validation renders, with depth);
* render: ``Pipeline.trace_benchmark``, the inference render of one camera;
* rebuild / move: ``Triangulation`` built from new points, and rebuilt incrementally
  after a small motion of all points, as the training loop does between steps;
* lookup: ``build_aabb_tree`` and ``nn`` over a point set.

The scenes are the ones that the bench and the tests use: "box" (uniform points),
"sphere" (a noisy shell in a box), "object" (a noisy superquadric surface in a box)
and "blobs" (Gaussian blobs inside a 1 / r^2 shell).  They are made on the GPU, and
their adjacency by ``Triangulation``, as a program has it.
"""

from __future__ import annotations

import math

import torch

import sdfoam_amd

INV_S = math.exp(0.3)  # the sharpness at the start of training
# walk steps per ray over the cube root of the points, as the scenes' cameras meet them
STEPS = {"box": 1.55, "sphere": 1.3, "object": 1.11, "blobs": 1.4}
FACES = 15.4  # neighbours of a point, on average
TETS = 6.7  # tetrahedra per point, on average
DTYPES = {"float32": torch.float32, "float16": torch.float16}


def _train(name, scene, points, width, height, rays, sh=3, mode="sdfoam", dtype="float32",
           quantiles=1, contribution=False, error=False, inv_s=INV_S, kind="train"):
    return {"name": name, "kind": kind, "scene": scene, "points": points, "width": width,
            "height": height, "rays": rays, "sh": sh, "mode": mode, "dtype": dtype,
            "quantiles": quantiles, "contribution": contribution, "error": error, "inv_s": inv_s}


def _render(name, scene, points, width, height, sh=3, mode="sdfoam", dtype="float32",
            model="pinhole", threshold=0.05):
    return {"name": name, "kind": "render", "scene": scene, "points": points, "width": width,
            "height": height, "sh": sh, "mode": mode, "dtype": dtype, "model": model,
            "threshold": threshold, "inv_s": INV_S}


def listed():
    return [
        # the headline: every ray of a 1600x1200 image through one million cells
        _train("train_image_1600x1200", "object", 1_000_000, 1600, 1200, 0, contribution=True),
        # a training step over random rays of 64 cameras, two depth quantiles, moved points
        _train("train_batch_1m", "blobs", 2_000_000, 960, 640, 1 << 20, quantiles=2),
        # the same early in a run or on a small scene: fewer points, a ragged batch, density mode
        _train("train_batch_65k", "blobs", 200_003, 641, 479, 65_537, sh=2, mode="standard",
               quantiles=2),
        # density mode over an image, with the per-point error that densification asks for
        _train("train_image_400", "sphere", 100_000, 400, 400, 0, mode="standard", error=True),
        # fp16 attributes, an image of odd sides, a sharp surface
        _train("train_image_fp16", "blobs", 300_007, 801, 601, 0, dtype="float16", quantiles=0,
               inv_s=50.0),
        # the smallest step: 4,104 cells, SH degree 0, 64x64 rays, where latency counts
        _train("train_image_64", "box", 4_104, 64, 64, 0, sh=0, contribution=True),
        # a validation render with depth of one camera of a large scene
        _train("eval_image_1297x840", "blobs", 3_000_000, 1297, 840, 0, kind="eval"),
        # the inference render: a full frame, and a small fisheye one
        _render("render_1600x1200", "object", 1_000_000, 1600, 1200),
        _render("render_small_fisheye", "sphere", 100_000, 321, 241, sh=1, mode="standard",
                model="fisheye", threshold=1e-3),
        # the adjacency from scratch, and after a small motion of every point
        {"name": "rebuild_1m", "kind": "rebuild", "scene": "object", "points": 1_000_000},
        {"name": "move_200k", "kind": "move", "scene": "blobs", "points": 200_003,
         "motion": 0.001},
        # nearest cells of many positions (queries of no common origin)
        {"name": "lookup_100k", "kind": "lookup", "scene": "object", "points": 1_000_000,
         "queries": 100_003},
    ]


def _log(rng, lo, hi):
    """A whole number, its logarithm uniform."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["train", "eval", "render", "rebuild", "move", "lookup"],
                       [11, 2, 3, 2, 1, 1])[0]
    scene = rng.choice(["box", "sphere", "object", "blobs"])
    if kind == "rebuild":
        return {"kind": kind, "scene": scene, "points": _log(rng, 4_000, 1_000_000)}
    if kind == "move":
        return {"kind": kind, "scene": scene, "points": _log(rng, 4_000, 400_000),
                "motion": rng.choice([0.0003, 0.001, 0.003])}
    if kind == "lookup":
        return {"kind": kind, "scene": scene, "points": _log(rng, 4_000, 2_000_000),
                "queries": _log(rng, 1, 200_000)}
    width = _log(rng, 64, 1600)
    height = max(48, min(1200, int(width * rng.uniform(0.55, 1.1))))
    points = _log(rng, 4_000, 1_000_000)
    sh = rng.choice([0, 1, 2, 3, 3, 3])
    mode = rng.choice(["sdfoam", "sdfoam", "standard"])
    dtype = rng.choice(["float32", "float32", "float32", "float16"])
    if kind == "render":
        case = _render("", scene, points, width, height, sh, mode, dtype,
                       rng.choice(["pinhole", "pinhole", "fisheye"]), rng.choice([0.05, 1e-3]))
    else:
        batch = rng.random() < 0.5
        if batch:
            width, height = 960, 640
        case = _train("", scene, points, width, height, _log(rng, 4_000, 1 << 20) if batch else 0,
                      sh, mode, dtype, rng.choice([0, 1, 1, 2]), rng.random() < 0.4,
                      kind == "train" and rng.random() < 0.25,
                      rng.choice([INV_S, INV_S, 10.0, 50.0]), kind)
        if dtype == "float16":
            # per-point sums over the rays leave fp16's range in the cells all rays cross
            case["contribution"] = case["error"] = False
    del case["name"]
    return case


# ---- scenes ---------------------------------------------------------------


def _unit(n, g):
    d = torch.randn((n, 3), generator=g, device="cuda", dtype=torch.float64)
    return d / d.norm(dim=1, keepdim=True)


def _uniform(shape, lo, hi, g):
    return torch.rand(shape, generator=g, device="cuda", dtype=torch.float64) * (hi - lo) + lo


def _spow(w, m):
    return w.sign() * w.abs().pow(m)


def _points(scene, n, g):
    """Unsorted points [n, 3] float32, and what the scene's SDF needs."""
    if scene == "box":
        x, more = _uniform((n, 3), -1.0, 1.0, g), None
    elif scene == "sphere":
        k = n * 4 // 5
        r = 0.5 + 0.02 * torch.randn((k, 1), generator=g, device="cuda", dtype=torch.float64)
        x, more = torch.cat([_unit(k, g) * r, _uniform((n - k, 3), -1.5, 1.5, g)]), None
    elif scene == "object":
        e = _uniform((2,), 0.5, 2.0, g)
        abc = _uniform((3,), 0.4, 0.6, g)
        k = n * 17 // 20
        eta, om = _uniform((k,), -math.pi / 2, math.pi / 2, g), _uniform((k,), -math.pi, math.pi, g)
        ce = _spow(eta.cos(), e[0])
        surf = torch.stack([ce * _spow(om.cos(), e[1]), ce * _spow(om.sin(), e[1]),
                            _spow(eta.sin(), e[0])], dim=1) * abc
        surf += 0.01 * torch.randn(surf.shape, generator=g, device="cuda", dtype=torch.float64)
        x, more = torch.cat([surf, _uniform((n - k, 3), -1.0, 1.0, g)]), (e, abc)
    else:
        centres = _unit(32, g) * _uniform((32, 1), 0.0, 1.0, g).pow(1.0 / 3.0)
        sigma = _uniform((32, 1), 0.05, 0.2, g)
        k = n * 3 // 5
        which = torch.randint(0, 32, (k,), generator=g, device="cuda")
        blob = centres[which] + sigma[which] * torch.randn((k, 3), generator=g, device="cuda",
                                                           dtype=torch.float64)
        r = blob.norm(dim=1, keepdim=True)
        blob = torch.where(r > 1.0, blob / (r * r), blob)  # back inside the unit ball
        x = torch.cat([blob, _unit(n - k, g) * _uniform((n - k, 1), 1.0, 16.0, g)])
        more = centres
    x = x[torch.randperm(n, generator=g, device="cuda")].float()
    return x, more


def _sdf(scene, p, more):
    p = p.double()
    r = p.norm(dim=1)
    if scene == "object":
        e, abc = more
        q = (p / abc).abs()
        f = (q[:, 0].pow(2 / e[1]) + q[:, 1].pow(2 / e[1])).pow(e[1] / e[0]) + q[:, 2].pow(2 / e[0])
        return r * (1.0 - f.pow(-e[0] / 2.0))
    if scene == "blobs":
        return torch.cdist(p, more).amin(dim=1) - 0.1
    return r - 0.5


CAMERA = {"box": (3.0, 50.0), "sphere": (3.0, 50.0), "object": (2.5, 40.0), "blobs": (4.0, 50.0)}


def _cameras(scene, count):
    """count camera frames (position, forward, right, up) [count, 3] around the scene."""
    dist, fov = CAMERA[scene]
    k = torch.arange(count, dtype=torch.float64) + 0.5
    z = (1.0 - 2.0 * k / count) if count > 1 else torch.full((1,), 0.5, dtype=torch.float64)
    phi = k * math.pi * (3.0 - math.sqrt(5.0)) + 0.3
    pos = dist * torch.stack([(1 - z * z).sqrt() * phi.cos(), (1 - z * z).sqrt() * phi.sin(), z], 1)
    fwd = -pos / pos.norm(dim=1, keepdim=True)
    world = torch.tensor([0.0, 0.0, 1.0], dtype=torch.float64).expand_as(fwd)
    right = torch.linalg.cross(fwd, world)
    right /= right.norm(dim=1, keepdim=True)
    up = torch.linalg.cross(right, fwd)
    return pos, fwd, right, up, math.radians(fov)


def _rays(scene, width, height, count, g):
    """Pinhole rays: [height, width, 6] of one camera, or `count` random ones of 64."""
    pos, fwd, right, up, fov = _cameras(scene, 64 if count else 1)
    frame = [t.cuda() for t in (pos, fwd, right, up)]
    if count:
        cam = torch.randint(0, 64, (count,), generator=g, device="cuda")
        px = torch.randint(0, width * height, (count,), generator=g, device="cuda")
        i, j = px % width, px // width
    else:
        cam = torch.zeros((), dtype=torch.int64, device="cuda")
        j, i = torch.meshgrid(torch.arange(height, device="cuda"),
                              torch.arange(width, device="cuda"), indexing="ij")
    u = (2.0 * i.double() / width - 1.0) * (width / height)
    v = 1.0 - 2.0 * j.double() / height
    p, f, r, w = (t[cam] for t in frame)
    d = f / math.tan(fov / 2) + u[..., None] * r + v[..., None] * w
    d = d / d.norm(dim=-1, keepdim=True)
    return torch.cat([p.expand_as(d), d], dim=-1).float().contiguous()


def _attributes(case, p, more, g):
    n, d = p.shape[0], 1 + 3 * (case["sh"] + 1) ** 2
    a = 0.3 * torch.randn((n, d), generator=g, device="cuda")
    if case["mode"] == "sdfoam":
        a[:, -1] = _sdf(case["scene"], p, more)
    else:
        logit = torch.randn((n,), generator=g, device="cuda")
        a[:, -1] = torch.nn.functional.softplus(logit, beta=10.0)
    return a.to(DTYPES[case["dtype"]])


def prepare(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 7919 + 1)
    raw, more = _points(case["scene"], case["points"], g)
    if case["kind"] == "rebuild":
        return {"case": case, "points": raw}
    if case["kind"] == "lookup":
        order = sdfoam_amd.Triangulation(raw).permutation().view(torch.int32).long()
        some = torch.randint(0, raw.shape[0], (case["queries"],), generator=g, device="cuda")
        near = raw[some] + 0.02 * torch.randn((case["queries"], 3), generator=g, device="cuda")
        return {"case": case, "points": raw[order].contiguous(), "queries": near}
    tri = sdfoam_amd.Triangulation(raw)
    p = raw[tri.permutation().view(torch.int32).long()].contiguous()
    adj, offs = tri.point_adjacency(), tri.point_adjacency_offsets()
    if case["kind"] == "move":
        _, radius = sdfoam_amd.farthest_neighbor(p, adj, offs)
        step = torch.randn(p.shape, generator=g, device="cuda") * (case["motion"] * radius)[:, None]
        return {"case": case, "points": p, "moved": p + step, "tri": tri}
    attrs = _attributes(case, p, more, g)
    s = {"case": case, "adj": adj, "offs": offs,
         "pipeline": sdfoam_amd.create_pipeline(case["sh"], case["dtype"])}
    if case["kind"] == "render":
        s["points"], s["attrs"] = p, attrs
        s["tree"] = sdfoam_amd.build_aabb_tree(p)
        s["inv_s"] = torch.tensor([case["inv_s"]], device="cuda")
        s["diff"] = sdfoam_amd.prefetch_adjacent_diff(p, adj, offs)[: adj.shape[0]]
        pos, fwd, right, up, fov = _cameras(case["scene"], 1)
        s["camera"] = {"position": pos[0].float().numpy(), "forward": fwd[0].float().numpy(),
                       "right": right[0].float().numpy(), "up": up[0].float().numpy(), "fov": fov,
                       "width": case["width"], "height": case["height"], "model": case["model"]}
        s["eye"] = pos[:1].float().cuda()
        return s
    if case["rays"]:
        # the points move between two rebuilds of the adjacency
        _, radius = sdfoam_amd.farthest_neighbor(p, adj, offs)
        p = p + torch.randn(p.shape, generator=g, device="cuda") * (0.01 * radius)[:, None]
    s["tree"] = sdfoam_amd.build_aabb_tree(p)
    rays = _rays(case["scene"], case["width"], case["height"], case["rays"], g)
    lead = tuple(rays.shape[:-1])
    learn = case["kind"] == "train"
    s["points"] = p.requires_grad_(learn)
    s["attrs"] = attrs.requires_grad_(learn)
    s["inv_s"] = torch.tensor([case["inv_s"]], device="cuda").requires_grad_(learn)
    s["rays"] = rays
    s["quantiles"] = None
    if case["quantiles"]:
        q = torch.rand(lead + (case["quantiles"],), generator=g, device="cuda")
        s["quantiles"] = q.sort(dim=-1, descending=True)[0].contiguous() \
            if case["quantiles"] > 1 else torch.full_like(q, 0.5)
    if learn:
        dt = DTYPES[case["dtype"]]
        s["grad_rgba"] = torch.randn(lead + (4,), generator=g, device="cuda").to(dt)
        s["grad_depth"] = None if s["quantiles"] is None else \
            torch.randn(s["quantiles"].shape, generator=g, device="cuda")
        s["ray_error"] = torch.rand(lead, generator=g, device="cuda").to(dt) \
            if case["error"] else None
    return s


# ---- one pass ---------------------------------------------------------------


def _ints(t):
    return t.view(torch.int32)


def _room(t, rows):
    """t with rows of -2 after its own up to a number that depends on the case alone."""
    out = torch.full((rows,) + t.shape[1:], -2, dtype=torch.int32, device="cuda")
    out[: t.shape[0]] = _ints(t)
    return out


def _tables(tri, n):
    return {"tets": _room(tri.tets(), 8 * n), "tet_adjacency": _room(tri.tet_adjacency(), 8 * n),
            "adjacency": _room(tri.point_adjacency(), 18 * n),
            "vert_to_tet": _ints(tri.vert_to_tet()),
            "offsets": _ints(tri.point_adjacency_offsets())}


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "rebuild":
        tri = sdfoam_amd.Triangulation(s["points"])
        return dict(_tables(tri, case["points"]), permutation=_ints(tri.permutation()))
    if kind == "move":
        # there and back, so that every pass starts from the same tetrahedra
        s["tri"].rebuild(s["moved"], incremental=True)
        there = _tables(s["tri"], case["points"])
        s["tri"].rebuild(s["points"], incremental=True)
        return {"there": there, "back": _tables(s["tri"], case["points"])}
    if kind == "lookup":
        tree = sdfoam_amd.build_aabb_tree(s["points"])
        return {"tree": tree, "nearest": _ints(sdfoam_amd.nn(s["points"], tree, s["queries"]))}
    if kind == "render":
        start = sdfoam_amd.nn(s["points"], s["tree"], s["eye"])
        image = torch.empty((case["height"], case["width"]), dtype=torch.uint32, device="cuda")
        s["pipeline"].trace_benchmark(
            s["points"], s["attrs"], s["adj"], s["offs"], s["diff"], s["camera"], start, image,
            weight_threshold=case["threshold"], alpha_mode=case["mode"], inv_s=s["inv_s"])
        return {"image": _ints(image)}
    with torch.set_grad_enabled(kind == "train"):
        start = sdfoam_amd.get_starting_point(s["rays"], s["points"], s["tree"])
        # the sixth output, alpha, holds one visiting ray's value per point: which one is
        # not determined, so it is not compared
        rgba, depth, contribution, steps, box, _ = sdfoam_amd.TraceRays.apply(
            s["pipeline"], s["points"], s["attrs"], s["adj"], s["offs"], s["rays"], start,
            s["quantiles"], case["contribution"], case["mode"] == "sdfoam", s["inv_s"])
    out = {"rgba": rgba, "depth": depth, "contribution": contribution, "steps": _ints(steps)}
    if kind == "train":
        wanted = [s["points"], s["attrs"]] + ([s["inv_s"]] if case["mode"] == "sdfoam" else [])
        box.ray_error = s["ray_error"]
        got = torch.autograd.grad([rgba] + ([] if depth is None else [depth]), wanted,
                                  [s["grad_rgba"]] + ([] if depth is None else [s["grad_depth"]]))
        out.update(zip(("points_grad", "attr_grad", "inv_s_grad"), got))
        out["point_error"] = box.point_error
        out["rgba"] = rgba.detach()
        out["depth"] = None if depth is None else depth.detach()
    return out


def work(case):
    n, kind = case["points"], case["kind"]
    if kind == "rebuild":
        return {"bytes": 12 * n + 4 * n * (8 * TETS + 2 + FACES + 1), "flops": n * TETS * 400}
    if kind == "move":
        return {"bytes": 2 * (12 * n + 2 * 4 * n * (8 * TETS) + 4 * n * (2 + FACES)),
                "flops": 2 * n * TETS * 200}
    if kind == "lookup":
        return {"bytes": 12 * n + 24 * 2 ** math.ceil(math.log2(n)) + 16 * case["queries"],
                "flops": 12 * n + case["queries"] * 400}
    d = 1 + 3 * (case["sh"] + 1) ** 2
    a = 2 if case["dtype"] == "float16" else 4
    rays = case.get("rays") or case["width"] * case["height"]
    steps = rays * STEPS[case["scene"]] * n ** (1.0 / 3.0)
    scene = n * (12 + a * d + 4 + 4 * FACES)
    walk = FACES * 24 + 6 * (case["sh"] + 1) ** 2 + 40
    if kind == "render":
        return {"bytes": scene + 8 * FACES * n + 4 * rays, "flops": steps * walk}
    q = case["quantiles"]
    out = rays * (4 * a + 4 + 8 * q) + (n * a if case["contribution"] else 0)
    if kind == "eval":
        return {"bytes": scene + rays * (24 + 4 * q) + out, "flops": steps * walk}
    grads = n * (12 + a * d) + rays * (4 * a + 4 * q)
    if case["error"]:
        grads += a * (rays + n)
    return {"bytes": scene + rays * (24 + 4 * q) + out + grads,
            "flops": steps * (walk + 6 * (case["sh"] + 1) ** 2 + 150)}


def tolerance(case):
    """Images, triangulations and lookups are whole numbers.  A trace's sums over rays have
    no order: twice the same pass differs by up to 1.2e-5 (2-norm) and 6e-4 (one value) in
    fp32, and by one rounding (2^-10) of some values in fp16."""
    if case["kind"] not in ("train", "eval"):
        return "exact"
    return {"rel": 1e-4, "max": 4e-3} if case["dtype"] == "float16" else {"rel": 5e-5, "max": 2.5e-3}


# ---- the trace in 64 bits -----------------------------------------------------


def _basis(degree, d):
    x, y, z = d.unbind(-1)
    one = torch.ones_like(x)
    b = [0.28209479177387814 * one]
    if degree > 0:
        b += [-0.4886025119029199 * y, 0.4886025119029199 * z, -0.4886025119029199 * x]
    if degree > 1:
        k = 1.0925484305920792
        b += [k * x * y, -k * y * z, 0.31539156525252005 * (2 * z * z - x * x - y * y),
              -k * x * z, k / 2 * (x * x - y * y)]
    if degree > 2:
        b += [-0.5900435899266435 * y * (3 * x * x - y * y), 2.890611442640554 * x * y * z,
              -0.4570457994644658 * y * (4 * z * z - x * x - y * y),
              0.3731763325901154 * z * (2 * z * z - 3 * x * x - 3 * y * y),
              -0.4570457994644658 * x * (4 * z * z - x * x - y * y),
              1.445305721320277 * z * (x * x - y * y),
              -0.5900435899266435 * x * (x * x - 3 * y * y)]
    return torch.stack(b, dim=-1)


def _face_grad(p, q, o, d):
    """d t / d p of the plane halfway between p and q."""
    fn = q - p
    num = (((p + q) / 2 - o) * fn).sum(-1, keepdim=True)
    dp = (fn * d).sum(-1, keepdim=True)
    return (num * d + dp * (o - p)) / (dp * dp)


def _walk(e, o, d, start, safe, visit):
    """The walk of rays through the cells: visit(ray, cell, next, t0, t1) at every step,
    which says which of those rays go on."""
    ray = torch.arange(start.shape[0], device="cuda")
    cell, t0 = start.clone(), torch.zeros(start.shape[0], dtype=torch.float64, device="cuda")
    for _ in range(1024):
        beg, deg = e["offs"][cell], e["offs"][cell + 1] - e["offs"][cell]
        own = torch.repeat_interleave(torch.arange(ray.shape[0], device="cuda"), deg)
        at = torch.arange(own.shape[0], device="cuda") - (deg.cumsum(0) - deg)[own] + beg[own]
        v = e["diff"][at]
        dp = (v * d[ray[own]]).sum(1)
        t = ((e["points"][cell[own]] + v / 2 - o[ray[own]]) * v).sum(1) / dp
        ok = (dp > 0) & (t > t0[own]) if safe else dp > 0
        t = torch.where(ok, t, math.inf)
        t1 = torch.segment_reduce(t, "min", lengths=deg, unsafe=True)
        at = torch.where(ok & (t == t1[own]), at.double(), math.inf)
        at = torch.segment_reduce(at, "min", lengths=deg, unsafe=True)
        live = t1 < math.inf
        ray, cell, t0, t1, at = (x[live] for x in (ray, cell, t0, t1, at))
        nxt = e["adj"][at.long()]
        step = t1 > t0
        go = torch.ones_like(step)
        go[step] = visit(ray[step], cell[step], nxt[step], t0[step], t1[step])
        ray, cell, t0 = ray[go], nxt[go], torch.maximum(t0, t1)[go]
        if not ray.shape[0]:
            return


def _add_rows(to, at, rows):
    """to[at] += rows, where many rows may go to one place: into copies of it first."""
    if not at.shape[0]:
        return
    places, which = torch.unique(at, return_inverse=True)
    copies = max(1, at.shape[0] // places.shape[0])
    turn = torch.arange(at.shape[0], device="cuda") % copies
    part = torch.zeros((places.shape[0] * copies,) + rows.shape[1:], dtype=rows.dtype, device="cuda")
    part.index_add_(0, which * copies + turn, rows)
    to[places] += part.view((-1, copies) + rows.shape[1:]).sum(1)


def _trace(e, s, lo, hi, out):
    case = s["case"]
    sdf, degree = case["mode"] == "sdfoam", case["sh"]
    f64 = {"dtype": torch.float64, "device": "cuda"}
    rays = s["rays"].view(-1, 6)[lo:hi].double()
    m = rays.shape[0]
    o, d = rays[:, :3], rays[:, 3:] / rays[:, 3:].norm(dim=1, keepdim=True)
    start, Y, inv_s = e["start"][lo:hi], _basis(degree, d), float(case["inv_s"])
    Q = case["quantiles"]
    q = s["quantiles"].view(-1, Q)[lo:hi].double() if Q else None
    attrs, P = e["attrs"], e["points"]
    T, C = torch.ones(m, **f64), torch.zeros((m, 3), **f64)
    qi = torch.zeros(m, dtype=torch.int64, device="cuda")
    depth = torch.full((m, Q), -1.0, **f64)
    crossed = torch.zeros(m, **f64)  # density mode: depth gradient over the crossed density

    def shade(r, c, t0, t1):
        row = attrs[c]
        last = row[:, -1]
        phi = torch.sigmoid(-inv_s * last)
        density = inv_s * phi * (1 - phi) if sdf else last
        alpha = 1 - torch.exp(-density * (t1 - t0))
        sh = row[:, :-1].view(r.shape[0], Y.shape[1], 3)
        rgb = (0.5 + (Y[r][:, :, None] * sh).sum(1)).clamp(min=0)
        if not sdf:
            rgb = torch.where(last[:, None] > 1e-6, rgb, 0.0)
        return last, phi, density, alpha, rgb

    def crossing(r, Tn, drop, j):
        hit = (qi[r] == j) & (Tn < q[r, j])
        return hit & (drop > 1e-12) if sdf else hit

    def forward(r, c, nxt, t0, t1):
        _, _, density, alpha, rgb = shade(r, c, t0, t1)
        w, Tr = T[r] * alpha, T[r]
        Tn = Tr * (1 - alpha)
        C[r] += w[:, None] * rgb
        if out["contribution"] is not None:
            _add_rows(out["contribution"].view(-1), c, w)
        for j in range(Q):
            k = crossing(r, Tn, Tr - Tn, j)
            rj, Tk = r[k], Tr[k]
            if sdf:
                frac = ((Tk - q[rj, j]) / (Tk - Tn[k])).clamp(0, 1)
                depth[rj, j] = t0[k] + frac * (t1 - t0)[k]
            else:
                depth[rj, j] = t0[k] + torch.log(Tk / q[rj, j]) / density[k]
                if e["learn"]:
                    crossed[rj] += e["grad_depth"][lo + rj, j] / density[k]
            qi[rj] += 1
        T[r] = Tn
        return Tn > 1e-7

    _walk(e, o, d, start, True, forward)
    out["rgba"][lo:hi, :3], out["rgba"][lo:hi, 3] = C, 1 - T
    if Q:
        out["depth"][lo:hi] = depth
    if not e["learn"]:
        return
    g4 = s["grad_rgba"].view(-1, 4)[lo:hi].double()
    # the backward reads the forward's rgba: rounded, where its type is fp16
    final = torch.cat([C, (1 - T)[:, None]], dim=1)
    if case["dtype"] == "float16":
        final = final.half().double()
    err = s["ray_error"].view(-1)[lo:hi].double() if case["error"] else None
    gd = e["grad_depth"][lo:hi] if Q else None
    T.fill_(1.0), C.zero_(), qi.zero_()
    g_logT = torch.zeros(m, **f64)
    prev = torch.full((m,), -1, dtype=torch.int64, device="cuda")
    prev_x, prev_g, cur_g = (torch.zeros((m, 3), **f64) for _ in range(3))

    def backward(r, c, nxt, t0, t1):
        last, phi, density, alpha, rgb = shade(r, c, t0, t1)
        Tr, dt, oma = T[r], t1 - t0, 1 - alpha
        Tn, w = Tr * oma, Tr * alpha
        C[r] += w[:, None] * rgb
        g, fin = g4[r], final[r]
        den = Tn + 1e-6 if sdf else Tr * (oma + 1e-6)
        da = Tr * ((rgb - (fin[:, :3] - C[r]) / den[:, None]) * g[:, :3]).sum(1)
        da += (1 - fin[:, 3]) * g[:, 3] / (oma + 1e-6)
        if sdf:
            da -= g_logT[r] / oma.clamp(min=1e-12)
        ds, dd, dt0 = da * dt * oma, da * density * oma, torch.zeros_like(dt)
        for j in range(Q):
            k = crossing(r, Tn, Tr - Tn, j)
            rj, gq = r[k], gd[r[k], j]
            if sdf:
                frac = ((Tr[k] - q[rj, j]) / (Tr[k] - Tn[k])).clamp(0, 1)
                dt0[k] += gq
                dd[k] += gq * frac
                some = (alpha[k] > 1e-12) & (Tr[k] > 1e-20)
                g_logT[rj] += torch.where(some, gq * dt[k] * q[rj, j] / (alpha[k] * Tr[k]), 0.0)
            else:
                dt0[k] += gq / density[k]
                ds[k] -= gq / density[k] * torch.log(Tr[k] / q[rj, j]) / density[k]
                crossed[rj] -= gq / density[k]
            qi[rj] += 1
        if not sdf and Q:
            rest = torch.where(qi[r] < Q, crossed[r], 0.0)
            ds -= dt * rest
            dd -= density * rest
        dt0 -= dd
        # positions: a cell's gradient is added one step late, the last two never are
        x, xn, px = P[c], P[nxt], prev_x[r]
        had = prev[r] >= 0
        prev_g[r] += torch.where(had[:, None], dt0[:, None] * _face_grad(px, x, o[r], d[r]), 0.0)
        cur = cur_g[r] + dt0[:, None] * _face_grad(x, px, o[r], d[r]) \
            + dd[:, None] * _face_grad(x, xn, o[r], d[r])
        _add_rows(out["points_grad"], prev[r][had], prev_g[r][had])
        prev_g[r], cur_g[r] = cur, dd[:, None] * _face_grad(xn, x, o[r], d[r])
        prev_x[r], prev[r] = x, c
        # attributes
        colour = torch.where(rgb > 0, g[:, :3] * w[:, None], 0.0)
        rows = (Y[r][:, :, None] * colour[:, None, :]).flatten(1)
        if sdf:
            slope = phi * (1 - phi)
            out["inv_s_grad"] += (ds * slope * (1 - inv_s * last * (1 - 2 * phi))).sum()
            ds = -ds * inv_s * inv_s * (1 - 2 * phi) * slope
        _add_rows(out["attr_grad"], c, torch.cat([rows, ds[:, None]], dim=1))
        if err is not None:
            _add_rows(out["point_error"].view(-1), c, w * err[r])
        T[r] = Tn
        return Tn > 1e-7

    _walk(e, o, d, start, sdf, backward)


def exact(case, seed):
    """The trace's outputs in float64, from the same inputs: None for the whole numbers.

    None also for the depths of random quantiles (some are crossed in a hull cell, whose far
    face lies anywhere) and for the gradients of a scene that ends in its own hull ("box", "sphere",
    "object") and of density mode: there a few rays carry the norm, those that meet a hull
    cell they stay in for thousands of lengths (all terms after it are differences of nearly
    equal colours over a transmittance near 0) or a depth quantile in a cell of nearly no
    density (a term over its square), and 32 bits leave no digit of those.  The same kernels
    give the gradients of "blobs", whose hull is far where nothing is dense."""
    if case["kind"] not in ("train", "eval"):
        return None
    s = prepare(case, seed)
    learn = case["kind"] == "train"
    with torch.no_grad():
        p, rays = s["points"].detach(), s["rays"]
        offs, adj = _ints(s["offs"]).long(), _ints(s["adj"]).long()
        own = torch.repeat_interleave(torch.arange(p.shape[0], device="cuda"), offs[1:] - offs[:-1])
        origins, which = torch.unique(rays.view(-1, 6)[:, :3], dim=0, return_inverse=True)
        near = torch.stack([(p - x).double().square().sum(1).argmin() for x in origins])
        e = {"points": p.double(), "attrs": s["attrs"].detach().double(), "offs": offs, "adj": adj,
             # the walk's planes have half-precision normals by definition
             "diff": (p[adj] - p[own]).half().double(), "start": near[which], "learn": learn}
        if learn and case["quantiles"]:
            e["grad_depth"] = s["grad_depth"].view(-1, case["quantiles"]).double()
        f64 = {"dtype": torch.float64, "device": "cuda"}
        n, lead, R = p.shape[0], tuple(rays.shape[:-1]), rays.numel() // 6
        out = {"rgba": torch.zeros((R, 4), **f64),
               "depth": torch.zeros((R, case["quantiles"]), **f64) if case["quantiles"] else None,
               "contribution": torch.zeros((n, 1), **f64) if case["contribution"] else None,
               "steps": None}
        if learn:
            out.update(inv_s_grad=torch.zeros(1, **f64), points_grad=torch.zeros((n, 3), **f64),
                       attr_grad=torch.zeros(s["attrs"].shape, **f64),
                       point_error=torch.zeros((n, 1), **f64) if case["error"] else None)
        for lo in range(0, R, 1 << 19):
            _trace(e, s, lo, min(R, lo + (1 << 19)), out)
        out["rgba"] = out["rgba"].view(lead + (4,))
        out["depth"] = out["depth"].view(lead + (1,)) if case["quantiles"] == 1 else None
    if learn and (case["scene"] != "blobs" or case["mode"] != "sdfoam"):
        out.update(points_grad=None, attr_grad=None)
        if case["mode"] == "sdfoam":
            out["inv_s_grad"] = None
        else:
            del out["inv_s_grad"]
    return out
