"""bench.py's host-side pieces: the CPU baseline's contract fields and the
one-GPU guard (no GPU needed)."""

from __future__ import annotations

import subprocess
import sys
from pathlib import Path

import pytest
import torch

import bench
from torchbvh_amd import _handles, _native, _query

ROOT = Path(__file__).resolve().parents[1]


def test_cpu_baseline_fields_on_the_small_config():
    import os

    w = bench.make_workload("cfg1")
    clouds = bench.job_clouds(w)
    assert len(clouds) == 1 and clouds[0][0].shape == (10_000, 3)
    r = bench.cpu_baseline(clouds, w["k"], 256)
    assert set(r) == {"value", "unit", "cores", "kind", "sample"}
    assert r["kind"] == "port" and r["unit"] == "queries/s"
    assert r["value"] > 0 and r["cores"] == len(os.sched_getaffinity(0))
    assert "brute force" in r["sample"] and "256 of 10000" in r["sample"]
    d = bench.cpu_port_dfs(clouds, w["k"], 0.05)
    assert set(d) == set(r) and d["value"] > 0 and "C oracle" in d["sample"]


def test_cpu_baseline_sample_extrapolates_by_pairs():
    """Ragged clouds are sampled at different fractions: the sample's time
    scales by (query, point) pairs."""
    import numpy as np

    rng = np.random.default_rng(1)
    clouds = [(rng.random((n, 3), dtype=np.float32), rng.random((m, 3), dtype=np.float32))
              for n, m in ((300, 50), (2000, 400))]
    r = bench.cpu_baseline(clouds, 4, 64)
    assert "114 of 450" in r["sample"]  # all 50 of the first cloud, 64 of the second


def test_query_sort_byte_formulas():
    assert bench.qsort_bytes(10, 3) == 10 * (12 + 4 + 4 * 16 + 4)
    assert bench.qschedule_bytes(10, 3) == 10 * (12 + 4 + 2 * 16 + 4)


def test_job_clouds_split_batched_and_ragged_workloads():
    w = bench.make_workload("cfg3")
    clouds = bench.job_clouds(w)
    assert len(clouds) == 32 and all(p.shape == (65_536, 3) for p, _ in clouds)
    w = bench.make_workload("cfg5")
    clouds = bench.job_clouds(w)
    off = w["offsets"].tolist()
    assert [len(p) for p, _ in clouds] == [b - a for a, b in zip(off, off[1:])]
    assert sum(len(q) for _, q in clouds) == w["queries"].shape[0]


def test_more_than_one_gpu_is_refused():
    r = subprocess.run([sys.executable, str(ROOT / "bench.py"), "--gpus", "2"],
                       capture_output=True, text=True, cwd=ROOT, timeout=120)
    assert r.returncode != 0
    assert "one GPU" in (r.stdout + r.stderr)


@pytest.mark.parametrize("kind,rows,order", [("single", 1 << 17, "input"), ("single", (1 << 17) + 1, "schedule"),
                                             ("single", 1 << 20, "fine"), ("batched", 1 << 20, "schedule"),
                                             ("batched", 1 << 21, "fine"), ("ragged", 1 << 21, "schedule")])
def test_timed_query_calls_are_those_of_query_knn(monkeypatch, kind, rows, order):
    """The timed step makes the binding calls of ``tb.query_knn``, with the same arguments."""
    made = []

    def record(name):
        def call(*args, **kwargs):
            made.append((name, [tuple(a.shape) if isinstance(a, torch.Tensor) else a for a in args], kwargs))
            found = torch.zeros(1, dtype=torch.int64)
            return (found, found) if name.startswith("query") else found
        return staticmethod(call)

    for name in ("morton_sort_queries_narrow", "morton_sort_queries_ragged", "safe_offsets", "query_knn_ragged",
                 "query_knn_batched_cached_bounds", "query_knn_batched_cached_bounds_ordered"):
        monkeypatch.setattr(_native._NativeOps, name, record(name))
    for check in ("check_cuda_f32", "check_source_points"):
        monkeypatch.setattr(_query, check, lambda *a, **kw: None)

    class Read:
        def __init__(self, *a, **kw):
            pass

        def values(self):
            return [0, rows // 2, rows]

    monkeypatch.setattr(_query, "OffsetsRead", Read)
    lead = {"single": (), "batched": (2,), "ragged": ()}[kind]
    n, k = 64, 16
    tree = {"node_aabbs": torch.zeros((*lead, 2 * n - 1, 6)), "sorted_indices": torch.zeros((*lead, n), dtype=torch.int64),
            "scene_min": torch.zeros((*lead, 3)), "scene_max": torch.zeros((*lead, 3)), "num_leaves": n,
            "num_real_nodes": 2 * n - 1, "dim": 3, "batch_size": 2, "batch_offsets": torch.tensor([0, 32, 64])}
    aux = {"accel": "the accel", "host_offsets": [0, 32, 64],
           "packed": {**tree, "node_offsets": torch.zeros(3, dtype=torch.int64)}}
    handle = {"single": _handles.BVHHandle, "batched": _handles.BatchedBVHHandle,
              "ragged": lambda data, aux: _handles.RaggedBVHHandle(data, [], aux)}[kind](tree, aux)
    queries = torch.zeros((2, rows // 2, 3) if kind == "batched" else (rows, 3))
    offsets = torch.tensor([0, rows // 2, rows])
    query = {"single": _query._query_knn_single, "batched": _query._query_knn_batched,
             "ragged": _query._query_knn_ragged}[kind]
    query(handle, queries, *((offsets, k) if kind == "ragged" else (k,)))
    public, made[:] = list(made), []
    bench.query_phases(kind, handle, queries, offsets, k, lambda: made.append("between"))
    assert bench.query_order(kind, 2 if kind == "batched" else 1, rows, k) == order
    assert made.pop(-2) == "between"
    assert made == public
