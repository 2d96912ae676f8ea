"""The radix sort without scan launches (clouds of at most 112 tiles of 4,096
rows, csrc/sort.hip) around its limit and its steps of eight tiles, for single,
batched and ragged calls, full and schedule orders, against a stable argsort of
the library's own codes (pinned elsewhere)."""

import numpy as np
import pytest
import torch

import oracle
import torchbvh_amd as tb
from torchbvh_amd._native import _C

pytestmark = pytest.mark.gpu
TILE, LIMIT = 4096, 112


def _expected(points, lo, hi):
    codes = _C.morton_codes(points, lo, hi).cpu().numpy()
    return np.argsort(codes, axis=1, kind="stable")


@pytest.mark.parametrize("B,n", [(1, 12_289), (3, 8 * TILE), (2, 8 * TILE + 1), (1, 16 * TILE + 5),
                                 (1, LIMIT * TILE), (1, LIMIT * TILE + 1), (2, 40_000)])
@pytest.mark.parametrize("dim", [2, 3])
def test_batched_order(B, n, dim):
    g = torch.Generator("cuda").manual_seed(n)
    p = (torch.rand((B, n, dim), generator=g, device="cuda") * 300).round() / 300  # equal codes too
    d = _C.build_bvh_batched_cooperative(p)
    want = _expected(p, d["scene_min"], d["scene_max"])
    assert np.array_equal(d["sorted_indices"].cpu().numpy(), want)
    full = _C.morton_sort_queries_narrow(p, d["scene_min"], d["scene_max"])
    assert np.array_equal(full.cpu().numpy(), want)
    sched = _C.morton_sort_queries_narrow(p, d["scene_min"], d["scene_max"], schedule=True)
    lo, hi = d["scene_min"].cpu().numpy(), d["scene_max"].cpu().numpy()
    assert np.array_equal(sched[0].cpu().numpy(), oracle.schedule_order(p[0].cpu().numpy(), lo[0], hi[0]))


@pytest.mark.parametrize("sizes", [[1, 5000, 4096, 30_000, 7], [200_000, 3, 100_000], [LIMIT * TILE, 1]])
def test_ragged_order(sizes):
    g = torch.Generator("cuda").manual_seed(len(sizes))
    off = [0, *np.cumsum(sizes).tolist()]
    p = torch.rand((off[-1], 3), generator=g, device="cuda")
    h = tb.build_bvh(p, batch_offsets=torch.tensor(off, device="cuda"))
    for b, child in enumerate(h._handles):
        rows = p[off[b]:off[b + 1]][None]
        want = _expected(rows, child["scene_min"][None].contiguous(), child["scene_max"][None].contiguous())
        assert np.array_equal(child["sorted_indices"].cpu().numpy(), want[0])
