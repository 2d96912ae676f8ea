"""Ragged calls are launched while their offsets travel to the host, over a
copy made safe on the device (tbvh_safe_offsets): the copy for valid and invalid
offsets, the errors and their order, and results equal to the build that waits."""

import pytest
import torch

import torchbvh_amd as tb
from torchbvh_amd._native import _C

pytestmark = pytest.mark.gpu


def _offsets(values):
    return torch.tensor(values, dtype=torch.int64, device="cuda")


@pytest.mark.parametrize("values", [[0, 3, 10], [0, 10], [1, 3, 10], [0, 3, 9], [0, 7, 3, 10], [0, 3, 3, 10],
                                    [0, 2**62, 10], [-2**62, 3, 10], [0] + list(range(1, 10)) + [10]])
def test_safe_offsets(values):
    B = len(values) - 1
    rises = values[0] == 0 and values[-1] == 10 and all(b > a for a, b in zip(values, values[1:]))
    want = values if rises else [i * 10 // B for i in range(B + 1)]
    assert _C.safe_offsets(_offsets(values), 10).tolist() == want


def test_safe_offsets_of_many_clouds():
    off = torch.arange(0, 5001, device="cuda")
    assert torch.equal(_C.safe_offsets(off, 5000), off)
    off[4000] = 17
    assert torch.equal(_C.safe_offsets(off, 5000), torch.arange(0, 5001, device="cuda"))


@pytest.mark.parametrize("bad,message", [([1, 500, 1000], "start at 0"), ([0, 500, 999], "final offset"),
                                         ([0, 500, 500, 1000], "strictly increasing"),
                                         ([0, 2**40, 1000], "strictly increasing"),
                                         ([0, -2**40, 1000], "strictly increasing")])
def test_invalid_values_are_refused(bad, message):
    p = torch.rand((1000, 3), device="cuda")
    with pytest.raises(ValueError, match=message):
        tb.build_bvh(p, batch_offsets=_offsets(bad))
    bvh = tb.build_bvh(p, batch_offsets=_offsets([0, 400, 700, 1000] if len(bad) == 4 else [0, 400, 1000]))
    with pytest.raises(ValueError, match=message):
        tb.query_knn(bvh, p, 4, query_offsets=_offsets(bad))
    # The offsets' error comes before the later checks'.
    with pytest.raises(ValueError, match=message):
        tb.query_knn(bvh, p, 4, query_offsets=_offsets(bad), source_points=p[:3])
    with pytest.raises(ValueError, match="batch size must match"):
        tb.query_knn(bvh, p, 4, query_offsets=_offsets([0, 10, 20, 30, 40, 1000]))
    with pytest.raises(ValueError, match="strictly increasing"):
        tb.query_knn(bvh, p[:1], 4, query_offsets=_offsets([0] * (len(bad) - 1) + [1]))


@pytest.mark.parametrize("sizes", [[5], [1, 1, 1], [4, 9000, 17, 40_000], [3] * 700, [200_000, 1]])
@pytest.mark.parametrize("dim", [2, 3])
def test_build_equals_the_one_that_waits(sizes, dim):
    off = [0]
    for n in sizes:
        off.append(off[-1] + n)
    p = torch.rand((off[-1], dim), device="cuda")
    got = tb.build_bvh(p, batch_offsets=_offsets(off))
    want = _C.build_bvh_ragged(p, _offsets(off), sizes, with_accel=True)
    for key in ("node_aabbs", "sorted_indices", "scene_min", "scene_max", "left_child_mem", "right_child_mem",
                "mem_to_leaf", "node_offsets"):
        assert torch.equal(got._aux["packed"][key], want[key]), key
    child, n0, n1 = got._handles[-1], want["host_node_offsets"][-2], want["host_node_offsets"][-1]
    assert torch.equal(child["node_aabbs"], want["node_aabbs"][n0:n1])
    assert torch.equal(child["scene_max"], want["scene_max"][-1])
    if min(sizes) >= 4:
        a = tb.query_knn(got, p, 4, query_offsets=_offsets(off))
        for i, n in enumerate(sizes):
            rows = p[off[i]:off[i + 1]].contiguous()
            for x, y in zip(a, tb.query_knn(tb.build_bvh(rows), rows, 4)):
                assert torch.equal(x[off[i]:off[i + 1]], y)
