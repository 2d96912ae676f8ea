"""Performance cases: the work that programs have this library do, through its
public entry points, from the smallest calls to the largest.

A case is a dict of plain values.  ``kind`` says which calls one pass makes:

- ``step``: build a BVH and answer one set of queries (single or batched),
  as ``with BVH(points) as bvh: bvh.knn(queries, k)``.
- ``tree``: the same through ``build_bvh`` / ``query_knn``, and the program
  also reads the tree's arrays.
- ``lookup``: queries against a geometry that the program keeps.
- ``ragged``: packed clouds of different sizes, build and queries.
- ``heads``: displaced multi-head queries with the neighbours' coordinates.
- ``train``: displaced interpolation, forward and backward.
- ``routed``: two trees per sample, each query sent to one of them.

Neighbour indices and squared distances are reproducible bit for bit (ties
go to the lower index, distances are one fixed chain of fp32 operations), so
every case but ``train`` compares exactly.
"""

from __future__ import annotations

import math

import torch

import torchbvh_amd as tb
from torchbvh_amd._native import _C

DEVICE = "cuda"

# Brute force in 64 bits stays under about 20 seconds up to this many
# (query, point) pairs.
EXACT_PAIRS = 4_000_000_000


def listed():
    return [
        # One small cloud per call, where launches and latency count: the
        # smallest row of the published benchmark.
        {"name": "step_10k_3d", "kind": "step", "batch": 1, "points": 10_000, "queries": 10_000, "dim": 3,
         "k": 4, "cloud": "uniform", "ask": "uniform", "rows": False},
        # A few queries per call against geometry that is kept for a whole
        # forward pass, with the neighbours' coordinates.
        {"name": "lookup_1k_of_50k", "kind": "lookup", "batch": 1, "points": 50_000, "queries": 1_000, "dim": 3,
         "k": 8, "cloud": "uniform", "ask": "uniform"},
        # A batch of small planar clouds (published benchmark row); the
        # program also reads the tree.
        {"name": "tree_16x10k_2d", "kind": "tree", "batch": 16, "points": 10_000, "queries": 10_000, "dim": 2,
         "k": 4, "cloud": "uniform", "ask": "uniform"},
        # The headline workload: one million points, one million queries.
        {"name": "step_1m_3d", "kind": "step", "batch": 1, "points": 1_048_576, "queries": 1_048_576, "dim": 3,
         "k": 16, "cloud": "uniform", "ask": "uniform", "rows": False},
        # A training batch of clustered clouds, queries near the points.
        {"name": "step_32x65k_clustered", "kind": "step", "batch": 32, "points": 65_536, "queries": 65_536,
         "dim": 3, "k": 16, "cloud": "clusters", "ask": "near", "rows": False},
        # Large planar data (maps, images): jittered self-queries.
        {"name": "step_4m_2d", "kind": "step", "batch": 1, "points": 4_194_304, "queries": 4_194_304, "dim": 2,
         "k": 8, "cloud": "uniform", "ask": "near", "rows": False},
        # A scanned surface: the neighbour graph of every point, odd size,
        # with the neighbours' coordinates (normals, covariances).
        {"name": "scan_200k_self", "kind": "step", "batch": 1, "points": 200_003, "queries": 200_003, "dim": 3,
         "k": 16, "cloud": "surface", "ask": "self", "rows": True},
        # Surface clouds of very different sizes packed in one call, queries
        # anywhere in each cloud's box.
        {"name": "ragged_64_surface", "kind": "ragged", "clouds": 64, "least": 1_000, "most": 200_000, "dim": 3,
         "k": 32, "cloud": "surface", "ask": "uniform"},
        # Volumetric samples of different sizes packed in one call (particle
        # and mesh-node data), neighbours of every point.
        {"name": "ragged_37_volume", "kind": "ragged", "clouds": 37, "least": 801, "most": 60_013, "dim": 3,
         "k": 8, "cloud": "uniform", "ask": "self"},
        # Displaced attention: four heads look around every point.
        {"name": "heads_4x65k_4", "kind": "heads", "batch": 4, "points": 65_536, "heads": 4, "dim": 3, "k": 8,
         "cloud": "uniform"},
        # A training step through displaced interpolation: output and the
        # gradient of the values.
        {"name": "train_2x16k_4x16", "kind": "train", "batch": 2, "points": 16_384, "heads": 4, "channels": 16,
         "dim": 3, "k": 8, "cloud": "uniform"},
        # Queries split between two trees, as an interpolation with an
        # inside and an outside region makes them.
        {"name": "routed_1m_of_2x512k", "kind": "routed", "batch": 1, "points": 524_288, "others": 524_288,
         "queries": 1_048_576, "dim": 3, "k": 16, "cloud": "uniform"},
    ]


def _log_int(rng, least, most):
    return int(round(math.exp(rng.uniform(math.log(least), math.log(most)))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "tree", "lookup", "ragged", "ragged", "heads", "train", "routed"])
    dim = rng.choice([2, 3, 3])
    k = rng.choice([4, 8, 16, 32])
    cloud = rng.choice(["uniform", "clusters", "surface"])
    if kind in ("step", "tree"):
        batch = rng.choice([1, 1, 2, 5, 16, 32])
        # Total work up to the listed ones': 4M rows in the plane with few
        # neighbours, 1M to 2M otherwise.
        most = 4_194_304 if dim == 2 and k <= 8 else (1_048_576 if k == 32 else 2_097_152)
        points = _log_int(rng, 1_000, most // batch)
        queries = points
        ask = rng.choice(["uniform", "near", "self"])
        if ask == "uniform":
            queries = min(_log_int(rng, max(points // 8, 500), points * 2), most // batch)
        case = {"kind": kind, "batch": batch, "points": points, "queries": queries, "dim": dim, "k": k,
                "cloud": cloud, "ask": ask}
        if kind == "step":
            case["rows"] = rng.random() < 0.3
        return case
    if kind == "lookup":
        points = _log_int(rng, 2_000, 500_000)
        return {"kind": kind, "batch": rng.choice([1, 1, 4]), "points": points,
                "queries": min(_log_int(rng, 100, 50_000), points), "dim": dim, "k": k, "cloud": cloud,
                "ask": rng.choice(["uniform", "near"])}
    if kind == "ragged":
        clouds = rng.randint(3, 64)
        least = _log_int(rng, 200, 2_000)
        most = _log_int(rng, 4 * least, 2_000_000 // clouds if clouds > 20 else 100_000)
        return {"kind": kind, "clouds": clouds, "least": least, "most": most, "dim": dim, "k": k,
                "cloud": cloud, "ask": rng.choice(["uniform", "near", "self"])}
    if kind == "heads":
        return {"kind": kind, "batch": rng.randint(1, 4), "points": _log_int(rng, 2_000, 65_536),
                "heads": rng.choice([1, 2, 4, 8]), "dim": dim, "k": rng.choice([4, 8, 16]), "cloud": cloud}
    if kind == "train":
        return {"kind": kind, "batch": rng.randint(1, 2), "points": _log_int(rng, 1_000, 20_000),
                "heads": rng.choice([1, 2, 4]), "channels": rng.choice([4, 8, 16, 32, 13]), "dim": dim,
                "k": rng.choice([4, 8, 16]), "cloud": cloud}
    points = _log_int(rng, 20_000, 524_288)
    return {"kind": kind, "batch": 1, "points": points, "others": _log_int(rng, 20_000, 524_288),
            "queries": _log_int(rng, 20_000, 1_048_576), "dim": dim, "k": rng.choice([4, 8, 16]), "cloud": cloud}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _generator(seed, device=DEVICE):
    return torch.Generator(device).manual_seed(int(seed))


def _cloud(shape, kind, g):
    """Points of `shape` (..., n, D): uniform in the unit box, eight Gaussian
    clusters of sigma 0.02, or a noisy surface (a torus; in the plane a
    circle of the same radius)."""
    lead, n, dim = shape[:-2], shape[-2], shape[-1]
    if kind == "uniform":
        return torch.rand(shape, generator=g, device=DEVICE)
    if kind == "clusters":
        centres = torch.rand(lead + (8, dim), generator=g, device=DEVICE)
        which = torch.randint(0, 8, lead + (n, 1), generator=g, device=DEVICE).expand(shape)
        return centres.gather(-2, which) + 0.02 * torch.randn(shape, generator=g, device=DEVICE)
    angle = torch.rand(lead + (n, 2), generator=g, device=DEVICE) * (2.0 * math.pi)
    theta, phi = angle[..., 0], angle[..., 1]
    if dim == 2:
        p = torch.stack((0.35 * torch.cos(theta), 0.35 * torch.sin(theta)), -1)
    else:
        ring = 0.35 + 0.1 * torch.cos(phi)
        p = torch.stack((ring * torch.cos(theta), ring * torch.sin(theta), 0.1 * torch.sin(phi)), -1)
    return p + 0.5 + 0.002 * torch.randn(shape, generator=g, device=DEVICE)


def _queries(points, count, kind, g):
    """Queries for `points` (..., n, D): uniform in the points' box, the
    points displaced by a little, or the points themselves."""
    if kind == "self":
        return points.clone()
    if kind == "near":
        sigma = 0.01 if points.size(-1) == 2 else 0.005
        return points + sigma * torch.randn(points.shape, generator=g, device=DEVICE)
    lo, hi = points.amin(-2, keepdim=True), points.amax(-2, keepdim=True)
    u = torch.rand(points.shape[:-2] + (count, points.size(-1)), generator=g, device=DEVICE)
    return lo + u * (hi - lo)


def _sizes(case):
    """Cloud sizes of a ragged case: fixed by the case (a program's data set
    keeps its sizes), spread evenly between the least and the most."""
    g = _generator(case["clouds"] * 7919 + case["least"] + case["most"], "cpu")
    return torch.randint(case["least"], case["most"] + 1, (case["clouds"],), generator=g).tolist()


def prepare(case, seed):
    g = _generator(seed)
    kind, dim = case["kind"], case["dim"]
    state = {"case": case}
    if kind in ("step", "tree", "lookup"):
        shape = (case["batch"], case["points"], dim)
        points = _cloud(shape, case["cloud"], g)
        queries = _queries(points, case["queries"], case["ask"], g)
        if kind == "step" and case["batch"] == 1:
            points, queries = points[0].contiguous(), queries[0].contiguous()
        if kind == "lookup" and queries.size(1) > case["queries"]:
            queries = queries[:, :case["queries"]].contiguous()
        state.update(points=points, queries=queries)
        if kind == "lookup":
            state["geometry"] = tb.PointGeometry(points)
    elif kind == "ragged":
        sizes = _sizes(case)
        clouds = [_cloud((n, dim), case["cloud"], g) for n in sizes]
        asked = [_queries(c, c.size(0), case["ask"], g) for c in clouds]
        offsets = [0]
        for n in sizes:
            offsets.append(offsets[-1] + n)
        state.update(points=torch.cat(clouds), queries=torch.cat(asked),
                     offsets=torch.tensor(offsets, dtype=torch.int64, device=DEVICE))
    elif kind in ("heads", "train"):
        b, n, h = case["batch"], case["points"], case["heads"]
        points = _cloud((b, n, dim), case["cloud"], g)
        moved = 0.02 * torch.randn((b, n, h, dim), generator=g, device=DEVICE)
        state.update(points=points, queries=points.unsqueeze(2) + moved)
        if kind == "train":
            values = torch.randn((b, n, h, case["channels"]), generator=g, device=DEVICE)
            state.update(values=values.requires_grad_(),
                         upstream=torch.randn(values.shape, generator=g, device=DEVICE))
    else:
        b = case["batch"]
        inside = _cloud((b, case["points"], dim), case["cloud"], g)
        outside = _cloud((b, case["others"], dim), case["cloud"], g)
        lo = torch.minimum(inside.amin(1, keepdim=True), outside.amin(1, keepdim=True))
        hi = torch.maximum(inside.amax(1, keepdim=True), outside.amax(1, keepdim=True))
        u = torch.rand((b, case["queries"], dim), generator=g, device=DEVICE)
        state.update(true=_C.build_bvh_batched_cooperative(inside), false=_C.build_bvh_batched_cooperative(outside),
                     true_points=inside, false_points=outside, queries=lo + u * (hi - lo),
                     routes=torch.rand((b, case["queries"]), generator=g, device=DEVICE) < 0.5)
    return state


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
_TREE_KEYS = ("node_aabbs", "sorted_indices", "scene_min", "scene_max", "left_child_mem", "right_child_mem",
              "mem_to_leaf")


def run(state):
    case = state["case"]
    kind, k = case["kind"], case["k"]
    if kind == "step":
        with tb.BVH(state["points"]) as bvh:
            return bvh.knn(state["queries"], k, source_points=state["points"] if case["rows"] else None)
    if kind == "tree":
        handle = tb.build_bvh(state["points"])
        found = tb.query_knn(handle, state["queries"], k)
        return tuple(found) + tuple(handle[key] for key in _TREE_KEYS)
    if kind == "lookup":
        geometry = state["geometry"]
        return tb.query_knn(geometry.bvh, state["queries"], k, source_points=geometry.points)
    if kind == "ragged":
        with tb.BVH(state["points"], batch_offsets=state["offsets"]) as bvh:
            return bvh.knn(state["queries"], k, query_offsets=state["offsets"])
    if kind == "heads":
        return tb.query_displaced_knn(state["points"], state["queries"], k)
    if kind == "train":
        out = tb.interpolate_displaced(state["points"], state["queries"], state["values"], k)
        (grad,) = torch.autograd.grad(out, state["values"], state["upstream"])
        return out.detach(), grad
    t, f = state["true"], state["false"]
    order = _C.morton_sort_routed_queries_batched(state["queries"], state["routes"], t["scene_min"],
                                                  t["scene_max"], f["scene_min"], f["scene_max"])
    indices, distances = _C.query_knn_routed_batched_cached_bounds_spatial(
        t["node_aabbs"], t["sorted_indices"], f["node_aabbs"], f["sorted_indices"], state["queries"],
        state["routes"], order, t["num_leaves"], t["num_real_nodes"], f["num_leaves"], f["num_real_nodes"],
        case["dim"], k)
    return order, indices, distances


# ---------------------------------------------------------------------------
# What a pass cannot do without: inputs read once, outputs written once; per
# neighbour found one distance.
# ---------------------------------------------------------------------------
def work(case):
    kind, dim, k = case["kind"], case["dim"], case["k"]
    if kind == "ragged":
        points = queries = sum(_sizes(case))
    elif kind in ("heads", "train"):
        points = case["batch"] * case["points"]
        queries = points * case["heads"]
    elif kind == "routed":
        points = case["batch"] * (case["points"] + case["others"])
        queries = case["batch"] * case["queries"]
    else:
        points = case["batch"] * case["points"]
        queries = case["batch"] * (case["queries"] if case["ask"] == "uniform" or kind == "lookup"
                                   else case["points"])
    total = 4 * dim * (points + queries) + 12 * k * queries
    flops = (3 * dim - 1) * k * queries
    if case.get("rows") or kind in ("lookup", "heads"):
        total += 4 * dim * k * queries
    if kind == "tree":
        n = case["points"]
        level = (n - 1).bit_length()
        nodes = 2 * n - 1 + bin((1 << level) - n).count("1")
        total += case["batch"] * (8 * dim * nodes + 8 * n) + 12 * nodes
    if kind == "routed":
        total += 9 * queries
    if kind == "train":
        # Indices and weights stay inside; values, upstream, output and
        # gradient pass once.
        total += 4 * 4 * case["channels"] * queries - 12 * k * queries
        flops += 2 * 2 * k * case["channels"] * queries
    return {"bytes": total, "flops": flops}


def tolerance(case):
    if case["kind"] == "train":
        # fp32 sums of k terms (forward) and of the rows that a point feeds
        # (backward), in any order.
        return {"rel": 1e-6, "max": 2e-5}
    return "exact"


# ---------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------
def _brute(points, queries, k):
    """Indices and squared distances (M, k) in 64 bits, nearest first."""
    p = points.double()
    rows = max(1, 60_000_000 // p.size(0))
    idx, dist = [], []
    for q in queries.double().split(rows):
        d = torch.zeros((q.size(0), p.size(0)), dtype=torch.float64, device=q.device)
        for a in range(p.size(1)):
            d += (q[:, a, None] - p[None, :, a]) ** 2
        near, at = torch.topk(d, k, dim=1, largest=False, sorted=True)
        idx.append(at)
        dist.append(near)
    return torch.cat(idx), torch.cat(dist)


def exact(case, seed):
    kind, k = case["kind"], case["k"]
    if kind in ("routed", "ragged"):
        return None
    pairs = case["batch"] * case["points"] * (case["points"] * case["heads"] if kind in ("heads", "train")
                                              else max(case["queries"], 1))
    if pairs > EXACT_PAIRS:
        return None
    state = prepare({**case, "kind": "tree"} if kind == "lookup" else case, seed)
    points, queries = state["points"].detach(), state["queries"]
    if kind == "lookup" and queries.size(1) > case["queries"]:
        queries = queries[:, :case["queries"]].contiguous()
    if kind in ("heads", "train"):
        b, n, h, dim = queries.shape
        found = [_brute(points[i], queries[i].reshape(n * h, dim), k) for i in range(b)]
        idx = torch.stack([f[0] for f in found]).reshape(b, n, h, k)
        d2 = torch.stack([f[1] for f in found]).reshape(b, n, h, k)
        if kind == "heads":
            return None, d2, None
        eps = 1e-12
        hit = d2 <= eps
        w = 1.0 / (d2 + eps)
        w = w / w.sum(-1, keepdim=True).clamp(min=eps)
        mean = hit.double() / hit.double().sum(-1, keepdim=True).clamp(min=1.0)
        w = torch.where(hit.any(-1, keepdim=True), mean, w)
        values = state["values"].detach().double()
        upstream = state["upstream"].double()
        out, grad = torch.zeros_like(values), torch.zeros_like(values)
        head = torch.arange(h, device=values.device).expand(n, h)
        for i in range(b):
            for r in range(k):
                at = idx[i, :, :, r]
                out[i] += w[i, :, :, r, None] * values[i][at, head]
                grad[i].index_put_((at, head), w[i, :, :, r, None] * upstream[i], accumulate=True)
        return out, grad
    if points.dim() == 2:
        _, d2 = _brute(points, queries, k)
    else:
        d2 = torch.stack([_brute(p, q, k)[1] for p, q in zip(points, queries)])
    if kind == "lookup":
        return None, d2, None
    if kind == "tree":
        return (None, d2) + (None,) * len(_TREE_KEYS)
    return (None, d2, None) if case["rows"] else (None, d2)
