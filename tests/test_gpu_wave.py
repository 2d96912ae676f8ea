"""k-NN with one wave per query (tbvh_knn_accel_wave, csrc/knn_wave.hip)
against the oracle and, on the same calls, the one-query-per-lane traversal,
bit for bit: cloud sizes around the edges of its 16-point blocks and of its
steps of 64 boxes (1,024 and 65,536 points), every k, both dimensions, ties,
clustered and far queries, neighbour rows and launch-order output."""

import numpy as np
import pytest
import torch

import oracle
import torchbvh_amd as tb
from torchbvh_amd import _native
from torchbvh_amd._native import _C

pytestmark = pytest.mark.gpu

LIMITS = ("WAVE_MAX_QUERIES", "WAVE_MAX_QUERIES_2D", "WAVE_MAX_QUERIES_2D_LARGE")


def _both(monkeypatch, call):
    """The call through the wave search and through the traversal."""
    out = []
    for limit in (1 << 30, 0):
        for name in LIMITS:
            monkeypatch.setattr(_native, name, limit)
        out.append(call())
    return out


def _cloud(n, dim, kind, seed):
    rng = np.random.default_rng(seed)
    if kind == "uniform":
        p = rng.random((n, dim))
    elif kind == "grid":  # many exact ties
        p = rng.integers(0, 9, (n, dim)) / 8.0
    elif kind == "clusters":
        p = rng.random((5, dim))[rng.integers(0, 5, n)] + 0.003 * rng.standard_normal((n, dim))
    else:  # a sphere queried from its centre: every box within the k-th distance
        v = rng.standard_normal((n, dim))
        p = v / np.linalg.norm(v, axis=1, keepdims=True)
    return p.astype(np.float32)


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("kind", ["uniform", "grid", "clusters", "sphere"])
@pytest.mark.parametrize("n", [4, 15, 16, 17, 33, 1023, 1024, 1025, 4097, 65_535, 65_537])
def test_wave_search_matches_oracle(monkeypatch, n, kind, dim):
    pts = _cloud(n, dim, kind, 100 * n + dim)
    rng = np.random.default_rng(n)
    q = np.concatenate([pts[:20], rng.random((20, dim)) * 1.4 - 0.2, np.zeros((1, dim)), 50 * rng.random((3, dim))])
    q = q.astype(np.float32)
    tp, tq = torch.from_numpy(pts).cuda(), torch.from_numpy(q).cuda()
    bvh = tb.build_bvh(tp)
    for k in (4, 8, 16, 32):
        if k > n:
            continue
        wave, plain = _both(monkeypatch, lambda: tb.query_knn(bvh, tq, k, source_points=tp))
        ei, ed = oracle.knn(pts, q, k)
        assert np.array_equal(wave[0].cpu().numpy(), ei)
        assert np.array_equal(wave[1].cpu().numpy().view(np.uint32), ed.view(np.uint32))
        assert torch.equal(wave[2], tp[wave[0]])
        for a, b in zip(wave, plain):
            assert torch.equal(a, b)


@pytest.mark.parametrize("dim", [2, 3])
def test_wave_search_batched_ordered_spatial_and_wide_rows(monkeypatch, dim):
    g = torch.Generator("cuda").manual_seed(7)
    pts = torch.rand((3, 2500, dim), generator=g, device="cuda")
    q = torch.rand((3, 301, dim), generator=g, device="cuda")
    d = _C.build_bvh_batched_cooperative(pts)
    order = _C.morton_sort_queries_narrow(q, d["scene_min"], d["scene_max"])
    args = (d["node_aabbs"], d["sorted_indices"], q)
    tail = (d["num_leaves"], d["num_real_nodes"], dim, 8)
    src = torch.rand((3, 2500, 7), generator=g, device="cuda")
    calls = [
        lambda: _C.query_knn_batched_cached_bounds(*args, *tail, source_points=src),
        lambda: _C.query_knn_batched_cached_bounds_ordered(*args, order, *tail),
        lambda: _C.query_knn_batched_cached_bounds_spatial(*args, order, *tail),
    ]
    for call in calls:
        for a, b in zip(*_both(monkeypatch, call)):
            assert torch.equal(a, b)


def test_wave_search_non_finite(monkeypatch):
    pts = _cloud(3000, 3, "uniform", 5)
    pts[17] = np.inf
    pts[18, 1] = -np.inf
    q = _cloud(64, 3, "uniform", 6)
    q[0] = np.nan
    q[1, 2] = np.inf
    q[2, 0] = -np.inf
    tp, tq = torch.from_numpy(pts).cuda(), torch.from_numpy(q).cuda()
    bvh = tb.build_bvh(tp)
    wave, plain = _both(monkeypatch, lambda: tb.query_knn(bvh, tq, 8))
    for a, b in zip(wave, plain):
        assert torch.equal(a, b)


# Queries near a shell's centre are nearly equidistant from all of it, so the
# traversal's waves pass their budget of iterations and give them up
# (tbvh_knn_*_tail); the wave search of the same call is the reference.
def _shell(n, dim, seed):
    g = torch.Generator("cuda").manual_seed(seed)
    v = torch.randn((n, dim), generator=g, device="cuda")
    return v / v.norm(dim=1, keepdim=True) * (1.0 + 1e-3 * torch.rand((n, 1), generator=g, device="cuda"))


def _centre(m, dim, seed):
    g = torch.Generator("cuda").manual_seed(seed)
    return 0.3 * torch.randn((m, dim), generator=g, device="cuda")


@pytest.mark.parametrize("dim,k", [(2, 4), (2, 32), (3, 8), (3, 16), (3, 32)])
@pytest.mark.parametrize("layout", ["batched", "rows", "ordered", "ragged", "grid"])
def test_given_up_queries(monkeypatch, layout, dim, k):
    pts = torch.stack([_shell(33_000, dim, s) for s in (1, 2)])
    m = 70_000 if layout == "grid" else 15_000  # more than 2^17 queries: the cell-block search's fallback
    q = torch.stack([_centre(m, dim, s) for s in (3, 4)])
    if layout == "ragged":
        off = torch.tensor([0, 33_000, 66_000 - 7], device="cuda")
        qoff = torch.tensor([0, 15_000 + 3, 30_000], device="cuda")
        bvh = tb.build_bvh(pts.reshape(-1, dim)[:-7].contiguous(), batch_offsets=off)
        call = lambda: tb.query_knn(bvh, q.reshape(-1, dim), k, query_offsets=qoff)  # noqa: E731
    else:
        d = _C.build_bvh_batched_cooperative(pts)
        args = (d["node_aabbs"], d["sorted_indices"], q)
        tail = (d["num_leaves"], d["num_real_nodes"], dim, k)
        order = _C.morton_sort_queries_narrow(q, d["scene_min"], d["scene_max"])
        if layout == "ordered":
            call = lambda: _C.query_knn_batched_cached_bounds_ordered(*args, order, *tail)  # noqa: E731
        else:
            src = pts if layout == "rows" else None
            call = lambda: _C.query_knn_batched_cached_bounds(*args, *tail, source_points=src)  # noqa: E731
    wave, plain = _both(monkeypatch, call)
    for a, b in zip(wave, plain):
        assert torch.equal(a, b)
    if layout == "batched":
        rows = torch.arange(0, m, 997, device="cuda")
        ei, ed = oracle.knn(pts[1].cpu().numpy(), q[1, rows].cpu().numpy(), k)
        assert np.array_equal(plain[0][1, rows].cpu().numpy(), ei)
        assert np.array_equal(plain[1][1, rows].cpu().numpy().view(np.uint32), ed.view(np.uint32))


def test_queries_are_given_up():
    """The tail entry point marks queries here, and its rows are the plain
    traversal's."""
    L = _native.load()
    pts, q = _shell(33_000, 3, 1)[None], _centre(30_000, 3, 3)[None]
    d = _C.build_bvh_batched_cooperative(pts, with_accel=True)
    ws = torch.zeros(_native._size(L.tbvh_knn_tail_workspace_size, 30_000, 3), dtype=torch.uint8, device="cuda")
    out = [(torch.empty((30_000, 16), dtype=torch.int64, device="cuda"),
            torch.empty((30_000, 16), dtype=torch.float32, device="cuda")) for _ in range(2)]
    p, stream = _native._ptr, _native._stream(pts.device)
    _native._check(L.tbvh_knn_accel_tail(p(d["accel"]), p(d["node_aabbs"]), d["num_real_nodes"], p(q), None, 1, 30_000,
                                         33_000, 3, 16, 0, None, 0, p(out[0][0]), p(out[0][1]), None, p(ws),
                                         ws.numel(), stream))
    _native._check(L.tbvh_knn_accel(p(d["accel"]), p(q), None, 1, 30_000, 33_000, 3, 16, p(out[1][0]), p(out[1][1]),
                                    stream))
    masks = ws[: (30_000 + 63) // 64 * 8].view(torch.int64)
    assert int((masks != 0).sum()) > 100
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])


@pytest.mark.parametrize("dim,k", [(2, 8), (3, 16)])
def test_given_up_routed_queries(dim, k):
    a, b = _shell(20_000, dim, 1)[None], 1.5 * _shell(9_000, dim, 2)[None]
    q = _centre(30_000, dim, 3)[None]
    routes = torch.arange(30_000, device="cuda")[None] % 3 == 0
    t, f = _C.build_bvh_batched_cooperative(a), _C.build_bvh_batched_cooperative(b)
    order = torch.arange(30_000, device="cuda")[None].contiguous()
    i, d2 = _C.query_knn_routed_batched_cached_bounds_spatial(
        t["node_aabbs"], t["sorted_indices"], f["node_aabbs"], f["sorted_indices"], q, routes, order,
        t["num_leaves"], t["num_real_nodes"], f["num_leaves"], f["num_real_nodes"], dim, k)
    for payload, sel, offset in ((t, routes[0], 0), (f, ~routes[0], 20_000)):
        qs = q[:, sel].contiguous()
        ei, ed = _C.query_knn_batched_cached_bounds(payload["node_aabbs"], payload["sorted_indices"], qs,
                                                    payload["num_leaves"], payload["num_real_nodes"], dim, k)
        assert torch.equal(i[0, sel], ei[0] + offset)
        assert torch.equal(d2[0, sel], ed[0])


@pytest.mark.parametrize("layout", ["batched", "ragged"])
@pytest.mark.parametrize("k", [16, 32])
def test_given_up_queries_among_nan_points(layout, k):
    """Points with a NaN coordinate are near on their other axes, in boxes that
    are not.  Here the traversal scans one eighth first, 16 near points and 15
    with a NaN y beside one far in y, gives the query up over the shell in the
    other eighths, and the boxes within its k-th distance hold fewer than k
    points: the rows must still be distinct points at their true distances."""
    rng = np.random.default_rng(1)
    v = rng.standard_normal((3000, 3))
    v = v / np.linalg.norm(v, axis=1, keepdims=True) * (1 + 1e-3 * rng.random((3000, 1)))
    nan = np.stack([-0.05 - 0.4 * rng.random(15), np.full(15, np.nan), -0.05 - 0.4 * rng.random(15)], 1)
    near = np.stack([-5e-4 - 0.05 * rng.random(16), -5e-4 - 0.05 * rng.random(16), -0.99 - 1e-4 * rng.random(16)], 1)
    near[0, :2] = -5e-4
    pts = np.concatenate([v[~(v < 0).all(1)], nan, [[-0.25, -1.0, -0.25]], near]).astype(np.float32)
    q = (-2e-3 + 5e-4 * rng.standard_normal((30_000, 3))).astype(np.float32)
    tp, tq = torch.from_numpy(pts).cuda(), torch.from_numpy(q).cuda()
    if layout == "ragged":
        offsets = torch.tensor([0, len(pts)], device="cuda"), torch.tensor([0, len(q)], device="cuda")
        idx, d2 = tb.query_knn(tb.build_bvh(tp, batch_offsets=offsets[0]), tq, k, query_offsets=offsets[1])
    else:
        idx, d2 = tb.query_knn(tb.build_bvh(tp), tq, k)
    idx, d2 = idx.cpu().numpy(), d2.cpu().numpy()
    assert (idx >= 0).all()
    assert (np.diff(np.sort(idx, axis=1), axis=1) > 0).all()
    assert (np.diff(d2, axis=1) >= 0).all()
    assert np.array_equal(d2, oracle.pair_distances(pts, q, idx))


def _marks(ws, total_q, dim, k, grid):
    """The work-groups whose traversal gave queries up, from a call's workspace
    (knn.hip: set_tail, grid_layout)."""
    up = lambda x: (x + 255) // 256 * 256  # noqa: E731
    groups = -(-(-(-total_q // 64)) // 8) * 8
    if not grid:
        masks = ws[: groups * 8].view(torch.int64).cpu()
        return int((masks[: total_q // 64] != 0).sum())
    seg = -(-(groups // 8) // 64) * 64
    list2 = ws.numel() - up(total_q * 4) - up(512 * seg * 4)
    list1 = list2 - up(512 * seg * 4)
    counts = ws[list1 - 2 * 512 * 32 * 4: list1].view(torch.int32).view(2, 512, 32)[:, :, 0].cpu()
    two_passes = dim == 3 and k in (8, 16)
    masks = ws[list1 if two_passes else list2:][: groups * 8].view(torch.int64).cpu()
    b = torch.arange(groups)
    sub, chunk = b % 8 * 64 + b // 8 % 64, b // 8 // 64
    return int((masks[chunk * 64 < counts[1 if two_passes else 0][sub]] != 0).sum())


@pytest.mark.parametrize("k", [8, 16, 32])
@pytest.mark.parametrize("layout", ["batched", "rows", "ordered", "spatial", "ragged", "grid", "routed", "routed grid"])
def test_queries_are_given_up_in_every_layout(monkeypatch, layout, k):
    """The tail runs in each of them, and the rows are the whole traversal's."""
    L, p, used = _native.load(), _native._ptr, []

    def in_kept_workspace(entry):
        def call(*args):  # (..., workspace, size, stream)
            used.append(torch.zeros(args[-2], dtype=torch.uint8, device="cuda"))
            return entry(*args[:-3], p(used[-1]), *args[-2:])
        return call

    for name in LIMITS:
        monkeypatch.setattr(_native, name, 0)
    for name in ("tail", "ragged_tail", "routed_tail", "grid", "routed_grid_spatial"):
        monkeypatch.setattr(L, f"tbvh_knn_accel_{name}", in_kept_workspace(getattr(L, f"tbvh_knn_accel_{name}")))
    grid = "grid" in layout
    m = 134_000 if grid else 30_000
    q = _centre(m, 3, 3)[None]
    order = torch.randperm(m, generator=torch.Generator().manual_seed(1)).cuda()[None].contiguous()
    idx, dist = torch.empty((m, k), dtype=torch.int64, device="cuda"), torch.empty((m, k), device="cuda")
    stream = _native._stream(q.device)
    if layout == "ragged":
        off, qoff = torch.tensor([0, 15_000, 33_000], device="cuda"), torch.tensor([0, 9_999, m], device="cuda")
        bvh = tb.build_bvh(_shell(33_000, 3, 1), batch_offsets=off)
        got = tb.query_knn(bvh, q[0], k, query_offsets=qoff)
        _native._check(L.tbvh_knn_accel_ragged(p(bvh._aux["accel"]), p(off), 33_000, p(q), p(qoff), None, 2, m, 3, k,
                                               p(idx), p(dist), stream))
    elif layout.startswith("routed"):
        routes = torch.arange(m, device="cuda")[None] % 3 == 0
        t, f = (_C.build_bvh_batched_cooperative(c[None], with_accel=True)
                for c in (_shell(33_000, 3, 1), 1.5 * _shell(34_000, 3, 2)))
        got = _C.query_knn_routed_batched_cached_bounds_spatial(
            t["node_aabbs"], t["sorted_indices"], f["node_aabbs"], f["sorted_indices"], q, routes, order,
            t["num_leaves"], t["num_real_nodes"], f["num_leaves"], f["num_real_nodes"], 3, k)
        _native._check(L.tbvh_knn_accel_routed_spatial(p(t["accel"]), p(f["accel"]), p(q), p(routes), p(order), 1, m,
                                                       33_000, 34_000, 3, k, p(idx), p(dist), stream))
    else:
        pts = _shell(33_000, 3, 1)[None]
        d = _C.build_bvh_batched_cooperative(pts, with_accel=True)
        tree, sizes = (d["node_aabbs"], d["sorted_indices"], q), (33_000, d["num_real_nodes"], 3, k)
        plain = L.tbvh_knn_accel
        if layout in ("ordered", "spatial"):
            call = getattr(_C, f"query_knn_batched_cached_bounds_{layout}")
            got = call(*tree, order, *sizes)
            plain = L.tbvh_knn_accel_spatial if layout == "spatial" else plain
        else:
            got = _C.query_knn_batched_cached_bounds(*tree, *sizes, source_points=pts if layout == "rows" else None)
        _native._check(plain(p(d["accel"]), p(q), p(order) if layout in ("ordered", "spatial") else None, 1, m, 33_000,
                             3, k, p(idx), p(dist), stream))
    assert torch.equal(got[0].reshape(m, k), idx) and torch.equal(got[1].reshape(m, k), dist)
    assert len(used) == 1 and _marks(used[0], m, 3, k, grid) > 100
