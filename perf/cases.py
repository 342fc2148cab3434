"""The work that a user of this library has it do, as measurable cases: queries of every kind on one mesh, a
rebuild, a batch of meshes, walk on stars, and the learned bound's training and seeded search, from calls of a few
thousand queries on a small mesh to 2^22 queries on 2^20 triangles.

    listed()             the cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  what a program holds before the call (scenes built, inputs on the GPU)
    run(state)           one pass through the public entry points; returns its outputs
    work(case)           the bytes and operations that the pass cannot do without
    exact(case, seed)    the outputs in 64 bits, where brute force gives them in a few seconds
"""
import functools
import math

import numpy as np
import torch

import snch_lbvh_amd as S
from snch_lbvh_amd import workloads as W

# a mesh is named by its generator and its triangle count: "icosphere" (20 * 4^level), "sphere" (a closed noised
# sphere) and "torus" (open along one meridian, noised: it has boundary edges)
NEAREST, SILHOUETTE, RAYS, SAMPLES = "nearest", "silhouette", "rays", "samples"
REBUILD, BATCH, WALKS, SEEDED, GRADIENT = "rebuild", "batch", "walks", "seeded", "gradient"


def listed():
    return [
        # interactive use (picking, snapping): a short list of points against a small mesh, bound by latency
        {"name": "nearest_sphere_1k", "kind": NEAREST, "mesh": "icosphere", "triangles": 20480, "queries": 1000},
        # the small configuration: 65,536 points in a cube around a noised icosphere of 20,480 triangles
        {"name": "nearest_sphere_64k", "kind": NEAREST, "mesh": "icosphere", "triangles": 20480, "queries": 65536},
        # a distance field over a large mesh
        {"name": "nearest_torus_4m", "kind": NEAREST, "mesh": "torus", "triangles": 1 << 20, "queries": 1 << 22},
        # silhouettes for an odd, small number of walks inside a mid-sized mesh, flipped orientation
        {"name": "silhouette_torus_10k", "kind": SILHOUETTE, "mesh": "torus", "triangles": 90000, "queries": 10007,
         "flip": True},
        # the headline: closest silhouettes on 2^20 triangles, 2^22 queries
        {"name": "silhouette_torus_4m", "kind": SILHOUETTE, "mesh": "torus", "triangles": 1 << 20,
         "queries": 1 << 22, "flip": False},
        # closest hits of rays in every direction from points in the padded box
        {"name": "rays_torus_4m", "kind": RAYS, "mesh": "torus", "triangles": 1 << 20, "queries": 1 << 22,
         "any_hit": False},
        # SampleTriangleInSphere with radii over three decades
        {"name": "samples_torus_4m", "kind": SAMPLES, "mesh": "torus", "triangles": 1 << 20, "queries": 1 << 22},
        # the tree built again, then one frame of rays through it
        {"name": "rebuild_torus_1m", "kind": REBUILD, "mesh": "torus", "triangles": 1 << 20, "queries": 65536},
        # meshes and query sets of uneven sizes answered by one batched launch
        {"name": "batch_24_meshes", "kind": BATCH, "meshes": 24, "most_triangles": 200000, "most_queries": 1 << 18},
        # a Laplace solve by walk on stars: half the torus Dirichlet, half Neumann, up to 64 steps
        {"name": "walks_torus_128k", "kind": WALKS, "triangles": 1 << 20, "walks": 1 << 17, "steps": 64},
        # the learned bound in use: predicted radii, then the seeded exact search
        {"name": "seeded_torus_1m", "kind": SEEDED, "triangles": 1 << 20, "queries": 1 << 20},
        # the learned bound in training: loss and gradient of all weights over one large set of points
        {"name": "gradient_512k", "kind": GRADIENT, "points": 1 << 19},
    ]


def _log_int(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi]; seldom a round number."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice([NEAREST, NEAREST, SILHOUETTE, SILHOUETTE, RAYS, SAMPLES, REBUILD, BATCH, WALKS, SEEDED,
                       GRADIENT])
    if kind == BATCH:
        return {"kind": kind, "meshes": rng.randint(2, 24), "most_triangles": _log_int(rng, 4000, 200000),
                "most_queries": _log_int(rng, 8192, 1 << 18)}
    if kind == WALKS:
        return {"kind": kind, "triangles": _log_int(rng, 20000, 1 << 20), "walks": _log_int(rng, 1000, 1 << 17),
                "steps": rng.choice([32, 64])}
    if kind == SEEDED:
        return {"kind": kind, "triangles": _log_int(rng, 20000, 1 << 20), "queries": _log_int(rng, 4000, 1 << 20)}
    if kind == GRADIENT:
        return {"kind": kind, "points": _log_int(rng, 4000, 1 << 19)}
    case = {"kind": kind, "mesh": rng.choice(["sphere", "torus", "torus"]), "triangles": _log_int(rng, 2000, 1 << 20),
            "queries": _log_int(rng, 1000, 65536 if kind == REBUILD else 1 << 22)}
    if kind == SILHOUETTE:
        case["flip"] = rng.random() < 0.5
    if kind == RAYS:
        case["any_hit"] = rng.random() < 0.5
    return case


@functools.lru_cache(maxsize=48)
def _mesh(name, triangles, seed):
    """Host arrays (vertices, triangles) of about that many triangles."""
    if name == "icosphere":
        return W.icosphere(int(round(math.log(triangles / 20, 4))), 0.02, seed)
    if name == "sphere":
        return W.uv_sphere(triangles, 0.02, seed)
    nv = max(4, int(round(math.sqrt(triangles / 4))))
    return W.cut_torus(max(8, int(round(triangles / (2 * nv)))), nv, seed=seed)


def _rng(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _box_points(g, V, n, pad=0.1):
    """n points uniform in the padded bounding box of V, on the GPU."""
    lo, hi = W.padded_box(V, pad)
    lo, ext = torch.tensor(lo, device="cuda"), torch.tensor(hi - lo, device="cuda")
    return (lo + ext * torch.rand(n, 3, generator=g, device="cuda", dtype=torch.float64)).float()


def _directions(g, n):
    d = torch.randn(n, 3, generator=g, device="cuda", dtype=torch.float64)
    return (d / d.norm(dim=1, keepdim=True)).float()


def _queries(case, V, seed):
    """Query points: the icosphere's in the cube [-1.5, 1.5]^3, else in the padded box."""
    g = _rng(seed)
    if case["mesh"] == "icosphere":
        return 3.0 * torch.rand(case["queries"], 3, generator=g, device="cuda") - 1.5
    return _box_points(g, V, case["queries"])


def _training_points(g, V, F, n, sigma=0.05):
    """Half uniform in the padded box, half near the surface (a triangle's centroid plus N(0, sigma))."""
    far = _box_points(g, V, n - n // 2)
    Vg, Fg = torch.from_numpy(V).cuda(), torch.from_numpy(F).cuda().long()
    t = torch.randint(0, Fg.shape[0], (n // 2,), generator=g, device="cuda")
    near = Vg[Fg[t]].mean(1) + sigma * torch.randn(n // 2, 3, generator=g, device="cuda")
    return torch.cat([far, near])


def _bound(V, seed):
    lo, hi = W.padded_box(V)
    return S.LearnedBound(lo.astype(np.float32), hi.astype(np.float32), sigma=4.0, seed=seed)


def _batch_sizes(case):
    """Triangle and query counts of a batch's meshes, uniform in their logarithms: the same for every seed."""
    r = np.random.default_rng(case["meshes"])
    span = lambda lo, hi: np.exp(r.uniform(math.log(lo), math.log(hi), case["meshes"])).astype(int)  # noqa: E731
    return span(1e3, case["most_triangles"]), span(2 ** 12, case["most_queries"])


@functools.lru_cache(maxsize=16)
def _batch_meshes(triangles, seed):
    """Closed noised spheres and open tori in turn, on a grid of places."""
    meshes = []
    for k, n in enumerate(triangles):
        V, F = _mesh("torus" if k % 2 else "sphere", n, 64 * seed + k)
        meshes.append((V + np.float32([3.0 * (k % 8), 3.0 * (k // 8), 0.0]), F))
    return meshes


def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case}
    if kind == BATCH:
        triangles, queries = _batch_sizes(case)
        meshes = _batch_meshes(tuple(int(n) for n in triangles), seed)
        st["scene"] = S.BatchScene(meshes).build_bvh()
        g = _rng(seed)
        st["q"] = torch.cat([_box_points(g, V, int(n)) for (V, _), n in zip(meshes, queries)])
        st["q_off"] = np.concatenate([[0], np.cumsum(queries)]).astype(np.uint32)
        return st
    if kind == WALKS:
        V, F = _mesh("torus", case["triangles"], seed)
        dirichlet, neumann = W.split_dirichlet_neumann(V, F)
        st["solver"] = S.WoSt(S.Scene(V, dirichlet).build_bvh(), S.Scene(V, neumann).build_bvh(), case["walks"])
        st["x"] = torch.from_numpy(W.torus_interior_points(case["walks"], seed=seed)).cuda()
        st["seed"] = seed
        return st
    if kind == SEEDED:
        V, F = _mesh("torus", case["triangles"], seed)
        st["scene"] = S.Scene(V, F).build_bvh()
        g = _rng(seed)
        st["q"] = _box_points(g, V, case["queries"])
        # the network as its user keeps it: trained once on the mesh's own silhouette distances
        pts = _training_points(g, V, F, 1 << 18)
        st["bound"] = _bound(V, seed).set_loss(0.95)
        st["bound"].train(pts, st["scene"].closest_silhouette(pts)[1], batch=16384, epochs=8)
        return st
    if kind == GRADIENT:
        V, F = _mesh("icosphere", 20480, seed)
        st["bound"] = _bound(V, seed).set_loss(0.95)
        st["x"] = _training_points(_rng(seed), V, F, case["points"])
        st["d"] = S.Scene(V, F).build_bvh().closest_point(st["x"])[1]
        return st
    V, F = _mesh(case["mesh"], case["triangles"], seed)
    st["scene"] = S.Scene(V, F).build_bvh()
    st["q"] = _queries(case, V, seed)
    if kind in (RAYS, REBUILD):
        st["d"] = _directions(_rng(seed + 1), case["queries"])
    if kind == SAMPLES:
        g = _rng(seed + 1)
        lo, hi = math.log(1e-3), math.log(0.5)
        st["r"] = torch.exp(lo + (hi - lo) * torch.rand(case["queries"], generator=g, device="cuda"))
        st["u"] = torch.rand(case["queries"], 3, generator=g, device="cuda")
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == NEAREST:
        return st["scene"].closest_point(st["q"])
    if kind == SILHOUETTE:
        return st["scene"].closest_silhouette(st["q"], flip=case["flip"])
    if kind == RAYS:
        hit, t, uv, idx = st["scene"].ray_intersect(st["q"], st["d"], any_hit=case["any_hit"])
        return (hit,) if case["any_hit"] else (hit, t, uv, idx)
    if kind == SAMPLES:
        return st["scene"].sample_in_sphere(st["q"], st["r"], st["u"])
    if kind == REBUILD:
        return st["scene"].build_bvh().ray_intersect(st["q"], st["d"])
    if kind == BATCH:
        return st["scene"].closest_silhouette(st["q"], st["q_off"])
    if kind == WALKS:
        return st["solver"].solve(st["x"], max_steps=case["steps"], eps=1e-3, seed=st["seed"])
    if kind == SEEDED:
        return st["scene"].closest_silhouette(st["q"], seed_radius=st["bound"].seed_radius(st["q"], 0.05, 0.0))
    return st["bound"].gradient(st["x"], st["d"])


# one tree in its smallest useful form: per triangle 36 B of vertices, per internal node two boxes (48 B) and two
# child references (8 B); cones (axis, angle, radius of both children) 40 B; 1.5 edges of 32 B each
_TREE, _CONES = 36 + 56, 40 + 48
_BOX_TEST, _CONE_TEST = 14, 40  # FP32 operations


def work(case):
    """Each input read once, each output written once; operations of a search that goes straight to its answer
    (both children's boxes, and cones, at every level of a balanced tree)."""
    kind = case["kind"]
    n, q = case.get("triangles", 0), case.get("queries", 0)
    levels = math.log2(max(2, n))
    if kind == NEAREST:
        return {"bytes": n * _TREE + q * 20, "flops": q * levels * 2 * _BOX_TEST}
    if kind == SILHOUETTE:
        return {"bytes": n * (_TREE + _CONES) + q * 20, "flops": q * levels * 2 * (_BOX_TEST + _CONE_TEST)}
    if kind == RAYS:
        return {"bytes": n * _TREE + q * (24 + (1 if case["any_hit"] else 17)), "flops": q * levels * 2 * 21}
    if kind == SAMPLES:
        return {"bytes": n * _TREE + q * 48, "flops": q * levels * 2 * 30}
    if kind == REBUILD:  # vertices and indices in; tree, cones and edge records out; then the rays
        return {"bytes": n * (18 + _TREE + _CONES) + n * _TREE + q * 41, "flops": n * 300 + q * levels * 42}
    if kind == BATCH:
        n, q = (float(x.sum()) for x in _batch_sizes(case))
        levels = math.log2(case["most_triangles"])
        return {"bytes": n * (_TREE + _CONES) + q * 20, "flops": q * levels * 2 * (_BOX_TEST + _CONE_TEST)}
    if kind == WALKS:  # about 16 steps a walk, each with the four queries
        return {"bytes": n * (2 * _TREE + _CONES) + case["walks"] * 16,
                "flops": case["walks"] * 16 * levels * 2 * (3 * _BOX_TEST + _CONE_TEST)}
    weights = 64 * 128 + 3 * 128 * 128 + 128
    if kind == SEEDED:
        return {"bytes": n * (_TREE + _CONES) + q * 24 + 2 * weights,
                "flops": q * (2 * weights + levels * 2 * (_BOX_TEST + _CONE_TEST))}
    return {"bytes": case["points"] * 16 + 10 * weights, "flops": case["points"] * 6 * weights}


# ------------------------------------------------------------------ 64 bits
_MOST_PAIRS = 4e9  # queries x primitives that brute force takes on in a few seconds


def _chunks(n_prims, n):
    step = max(1, int(4e7) // max(1, n_prims))
    return [(k, min(n, k + step)) for k in range(0, n, step)]


def _segment(p, a, b):
    """Closest points of the segments a b to p, and the vectors from them to p."""
    u = b - a
    t = (((p - a) * u).sum(-1) / (u * u).sum(-1)).clamp(0, 1)
    return p - (a + t[..., None] * u)


def _nearest64(V, F, q):
    a, b, c = (V[F[:, k]] for k in range(3))
    n = torch.linalg.cross(b - a, c - a)
    n = n / n.norm(dim=1, keepdim=True)
    out = []
    for lo, hi in _chunks(4 * len(F), len(q)):
        p = q[lo:hi, None, :]
        d2 = torch.stack([(_segment(p, x, y) ** 2).sum(-1) for x, y in ((a, b), (b, c), (c, a))]).amin(0)
        h = ((p - a) * n).sum(-1)
        s = p - h[..., None] * n
        inside = torch.ones_like(h, dtype=torch.bool)
        for x, y in ((a, b), (b, c), (c, a)):
            inside &= (torch.linalg.cross((y - x).expand_as(s), s - x) * n).sum(-1) >= 0
        out.append(torch.where(inside, torch.minimum(d2, h * h), d2).amin(1).sqrt())
    return torch.cat(out)


def _edges(V, F):
    """Unique edges: end points and the unit normals of their two faces (has2: whether there are two)."""
    n = torch.linalg.cross(V[F[:, 1]] - V[F[:, 0]], V[F[:, 2]] - V[F[:, 0]])
    n = n / n.norm(dim=1, keepdim=True)
    e = torch.cat([F[:, [0, 1]], F[:, [1, 2]], F[:, [2, 0]]])
    face = torch.arange(len(F), device=F.device).repeat(3)
    key = e.amin(1) * len(V) + e.amax(1)
    # the face that runs from the lower to the higher vertex first
    order = torch.argsort(2 * key + (e[:, 0] > e[:, 1]).long())
    key, face = key[order], face[order]
    head = torch.ones_like(key, dtype=torch.bool)
    head[1:] = key[1:] != key[:-1]
    first = head.nonzero()[:, 0]
    second = (first + 1).clamp(max=len(key) - 1)
    has2 = (second > first) & (key[second] == key[first])
    lo, hi = key[first] // len(V), key[first] % len(V)
    return V[lo], V[hi], n[face[first]], n[face[second]], has2


def _silhouette64(V, F, q, flip):
    a, b, n0, n1, has2 = _edges(V, F)
    sign, eps = (1.0 if flip else -1.0), 1e-3
    ed = (b - a) / (b - a).norm(dim=1, keepdim=True)
    angle = torch.atan2((ed * torch.linalg.cross(n0, n1)).sum(1), (n0 * n1).sum(1))
    out = []
    for lo, hi in _chunks(2 * len(a), len(q)):
        v = _segment(q[lo:hi, None, :], a, b)
        d = v.norm(dim=-1)
        d0, d1 = (v * n0).sum(-1), (v * n1).sum(-1)
        sil = torch.where(d0.abs() <= eps, sign * d1 > eps,
                          torch.where(d1.abs() <= eps, sign * d0 > eps, d0 * d1 < 0))
        sil = torch.where(d <= eps, sign * angle > eps, sil) | ~has2
        out.append(torch.where(sil, d, math.inf).amin(1))
    return torch.cat(out)


def _rays64(V, F, o, d):
    v0, e1, e2 = V[F[:, 0]], V[F[:, 1]] - V[F[:, 0]], V[F[:, 2]] - V[F[:, 0]]
    out = []
    for lo, hi in _chunks(4 * len(F), len(o)):
        oo, dd = o[lo:hi, None, :], d[lo:hi, None, :]
        h = torch.linalg.cross(dd.expand(-1, len(F), 3), e2.expand(hi - lo, -1, 3))
        det = (e1 * h).sum(-1)
        s = oo - v0
        u = (s * h).sum(-1) / det
        q = torch.linalg.cross(s, e1.expand_as(s))
        v, t = (dd * q).sum(-1) / det, (e2 * q).sum(-1) / det
        ok = (det.abs() >= 2.0 ** -23) & (u >= 0) & (v >= 0) & (u + v <= 1) & (t >= 0)
        out.append(torch.where(ok, t, math.inf).amin(1))
    return torch.cat(out)


def _gradient64(st):
    theta, four, frame = st["bound"].params()
    th = torch.from_numpy(theta).cuda().double().requires_grad_(True)
    B = torch.from_numpy(four.reshape(32, 3)).cuda().double()
    c, inv, inv_d = (torch.tensor(frame[k], device="cuda").double() for k in (slice(0, 3), slice(3, 6), 6))
    x, d = st["x"].double(), st["d"].double()
    total = 0.0
    for lo, hi in [(k, min(len(x), k + 65536)) for k in range(0, len(x), 65536)]:
        f = (x[lo:hi] - c) * inv @ B.T
        a = torch.cat([f.sin(), f.cos()], 1)
        at = 0
        for k in (64, 128, 128, 128):
            w, b = th[at:at + 128 * k].reshape(128, k), th[at + 128 * k:at + 128 * k + 128]
            a = torch.nn.functional.silu(a @ w.T + b)
            at += 128 * k + 128
        err = a @ th[at:at + 128] + th[at + 128] - ((d[lo:hi] * inv_d).clamp(max=1.0) + 1e-3).log()
        loss = (2.0 * torch.where(err < 0, 0.95, 1.0 - 0.95) * err * err).sum() / len(x)
        loss.backward()
        total += float(loss)
    return th.grad.cpu().numpy(), total


def exact(case, seed):
    kind = case["kind"]
    if kind == GRADIENT:
        return _gradient64(prepare(case, seed))
    if kind not in (NEAREST, SILHOUETTE, RAYS) or case["triangles"] * case["queries"] > _MOST_PAIRS:
        return None
    V, F = _mesh(case["mesh"], case["triangles"], seed)
    q = _queries(case, V, seed).double()
    V, F = torch.from_numpy(V).cuda().double(), torch.from_numpy(F).cuda().long()
    if kind == NEAREST:
        return None, _nearest64(V, F, q)
    if kind == SILHOUETTE:
        return None, _silhouette64(V, F, q, case["flip"])
    if case["any_hit"]:
        return None
    return None, _rays64(V, F, q, _directions(_rng(seed + 1), case["queries"]).double()), None, None
