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
