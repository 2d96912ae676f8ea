"""The small-cloud sort's bins (csrc/small.hip) at the sizes where they change:
runs of equal codes around the count that sends a cloud to the stable passes
(32), runs that share a bin but not a code, clusters far denser than a bin,
and one bin for a whole cloud, in row order of every kind."""

import numpy as np
import pytest
import torch

import oracle
import torchbvh_amd as tb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("n", [300, 4096, 4097, 12_288])
@pytest.mark.parametrize("kind", ["run31", "run32", "run33", "run34", "run97", "near", "clusters", "outlier", "line"])
def test_order_matches_oracle(kind, n, dim):
    rng = np.random.default_rng(n + 7 * dim)
    p = rng.random((n, dim))
    if kind.startswith("run"):  # every point of a run at one place
        run = int(kind[3:])
        p[: 2 * run] = np.repeat(p[[0, run]], run, axis=0)
    elif kind == "near":  # codes that differ in their last bits only
        p[:200] = p[0] + rng.integers(0, 3, (200, dim)) / (1024 if dim == 3 else 65536)
    elif kind == "clusters":
        p = rng.random((4, dim))[rng.integers(0, 4, n)] + 1e-3 * rng.standard_normal((n, dim))
    elif kind == "outlier":  # one bin holds all but one
        p *= 1e-4
        p[n // 2] = 1.0
    else:
        p[:, 1:] = 0.5
    p = p[rng.permutation(n)].astype(np.float32)
    got, ref = tb.build_bvh(torch.from_numpy(p).cuda()), oracle.build(p)
    assert np.array_equal(got["sorted_indices"].cpu().numpy(), ref["sorted_indices"])
    assert np.array_equal(got["node_aabbs"].cpu().numpy().view(np.uint32), ref["node_aabbs"].view(np.uint32))
