"""The finer query schedule (tbvh_schedule_queries_fine): a permutation of every
cloud's queries whose sort tiles follow the keys' top 16 bits and are nearly in
order of 24, for sizes around the sort's tiles and the small sort's limit,
skewed queries, and the same search results."""

import numpy as np
import pytest
import torch

import torchbvh_amd as tb
from torchbvh_amd import _query
from torchbvh_amd._native import _C

pytestmark = pytest.mark.gpu


def _queries(B, M, dim, kind):
    g = torch.Generator("cuda").manual_seed(M + dim)
    q = torch.rand((B, M, dim), generator=g, device="cuda")
    if kind == "clusters":
        q = 0.5 + 1e-3 * (q - 0.5) + (torch.arange(M, device="cuda") % 3 == 0)[:, None] * 0.3
    elif kind == "same":
        q[:] = 0.25
        q[:, 0] = 0.9
    return q


@pytest.mark.parametrize("B,M", [(1, 1), (2, 12_288), (2, 12_289), (1, 4 * 4096), (3, 4 * 4096 + 1), (1, 500_003)])
@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("kind", ["uniform", "clusters", "same"])
def test_order(B, M, dim, kind):
    q = _queries(B, M, dim, kind)
    lo, hi = torch.zeros((B, dim), device="cuda"), torch.ones((B, dim), device="cuda")
    for k in (8, 32):  # Morton, Hilbert
        order = _C.morton_sort_queries_narrow(q, lo, hi, schedule=True, fine=k)
        assert torch.equal(order.sort(1)[0], torch.arange(M, device="cuda").expand(B, M))
        for _ in range(3):  # every call gives the same
            assert torch.equal(order, _C.morton_sort_queries_narrow(q, lo, hi, schedule=True, fine=k))
        if k == 8:
            bits = 30 if dim == 3 else 32
            codes = _C.morton_codes(q, lo, hi).gather(1, order)
            # Tiles hold the rows that the 16-bit order gives them ...
            top = codes >> (bits - 16)
            for t in range(0, M, 4096):
                top[:, t:t + 4096] = top[:, t:t + 4096].sort(1)[0]
            assert bool((top.diff(dim=1) >= 0).all())
            # ... nearly in order of the finer bits.
            if kind == "uniform" and M > 10_000:
                assert float(((codes >> (bits - 24)).diff(dim=1) >= 0).float().mean()) > 0.8


@pytest.mark.parametrize("k", [8, 32])
def test_search_results_do_not_depend_on_it(monkeypatch, k):
    p, q = _queries(2, 70_000, 3, "uniform"), _queries(2, 70_001, 3, "clusters")
    bvh = tb.build_bvh(p)
    want = tb.query_knn(bvh, q, k)
    monkeypatch.setattr(_query, "FINE_MIN_QUERIES", 1)
    for a, b in zip(want, tb.query_knn(bvh, q, k)):
        assert np.array_equal(a.cpu().numpy(), b.cpu().numpy())
