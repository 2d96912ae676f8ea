"""Multi-head displaced queries on top of the batched build and k-NN.

Mirrors the reference's helpers (torchbvh/_multihead.py:38-190): every
sample's points ``pos: (B, N, D)`` get one BVH; the per-point, per-head
query positions ``q: (B, N, H, D)`` are flattened to ``(B, N*H, D)`` and
answered by the Morton-ordered batched k-NN; results are reshaped back.
Names, argument checks and their messages follow the reference; the k-NN
underneath is this library's (exact, ties to the lower index).
"""

from __future__ import annotations

import torch

from ._constants import EXACT_DISTANCE_EPSILON, SUPPORTED_DIMS
from ._handles import scoped_bvh
from ._native import _C
from ._query import _build_bvh_batched, _query_knn_batched
from ._validation import check_cuda_f32, dense, dense_offsets

__all__ = ["query_displaced_knn", "gather_neighbor_values", "interpolate_displaced"]


_NOT_LOCAL = "gather_neighbor_values: indices must be local source indices"


def _check_displaced(pos: torch.Tensor, q: torch.Tensor, op: str) -> None:
    """Shape, dtype and device checks of the displaced-query helpers
    (reference order and messages: _multihead.py:17-35)."""
    if pos.dim() != 3:
        raise ValueError(f"{op}: pos must have shape (B, N, D)")
    if q.dim() != 4:
        raise ValueError(f"{op}: q must have shape (B, N, H, D)")
    if pos.size(2) not in SUPPORTED_DIMS:
        raise ValueError(f"{op}: D must be 2 or 3")
    checks = (
        (q.size(0) == pos.size(0), "q batch size must match pos"),
        (q.size(1) == pos.size(1), "q point dimension must match pos"),
        (q.size(3) == pos.size(2), "q last dimension must match pos"),
        (q.size(2) >= 1, "q must contain at least one head"),
    )
    for ok, message in checks:
        if not ok:
            raise ValueError(f"{op}: {message}")
    check_cuda_f32(op, pos, "pos")
    check_cuda_f32(op, q, "q")
    if pos.device != q.device:
        raise ValueError(f"{op}: pos and q must be on the same device")


def query_displaced_knn(pos: torch.Tensor, q: torch.Tensor, k: int = 8, *,
                        return_positions: bool = True):
    """k nearest points of ``pos[b]`` to every displaced query ``q[b, n, h]``.

    Returns local indices and squared distances of shape ``(B, N, H, k)``
    and, with ``return_positions``, the neighbours' coordinates
    ``(B, N, H, k, D)``."""
    _check_displaced(pos, q, "query_displaced_knn")
    pos = dense(pos)
    q = dense(q)
    B, N, H, D = q.shape
    queries = q.reshape(B, N * H, D).contiguous()
    sources = pos.detach().contiguous()
    with scoped_bvh(_build_bvh_batched, sources) as bvh:
        out = _query_knn_batched(bvh, queries, k,
                                 source_points=sources if return_positions else None,
                                 sort_queries=True)
    shapes = ((B, N, H, k), (B, N, H, k), (B, N, H, k, D))
    return tuple(t.reshape(shape).contiguous() for t, shape in zip(out, shapes))


def gather_neighbor_values(values: torch.Tensor, indices: torch.Tensor) -> torch.Tensor:
    """``out[b, n, h, j] = values[b, indices[b, n, h, j], h]``: per-head
    values of each neighbour, from the matching head only."""
    op = "gather_neighbor_values"
    if values.dim() != 4:
        raise ValueError(f"{op}: values must have shape (B, N, H, Ch)")
    if indices.dim() != 4:
        raise ValueError(f"{op}: indices must have shape (B, N, H, k)")
    for axis, what in ((0, "batch size"), (1, "point dimension"), (2, "head dimension")):
        if values.size(axis) != indices.size(axis):
            raise ValueError(f"{op}: indices {what} must match values")
    if values.size(3) < 1:
        raise ValueError(f"{op}: values must have at least one channel")
    check_cuda_f32(op, values, "values")
    if indices.dtype != torch.int64:
        raise ValueError(f"{op}: indices must be int64")
    if values.device != indices.device:
        raise ValueError(f"{op}: values and indices must be on the same device")
    values = dense(values)
    indices = dense_offsets(indices)
    if indices.numel() > 0:
        lo, hi = torch.aminmax(indices)
        if int(lo) < 0 or int(hi) >= values.size(1):
            raise ValueError(_NOT_LOCAL)
    return _gather(values, indices)


def _gather(values: torch.Tensor, indices: torch.Tensor) -> torch.Tensor:
    B, _, H, _ = values.shape
    batch = torch.arange(B, device=values.device).view(B, 1, 1, 1)
    head = torch.arange(H, device=values.device).view(1, 1, H, 1)
    return values[batch, indices, head]


def _combine(neighbours: torch.Tensor, weights: torch.Tensor, exact: torch.Tensor) -> torch.Tensor:
    """(B, N, H, k, Ch) neighbours to their weighted means, or those of a row's
    exact hits.  Accumulated neighbour rank by neighbour rank, the reference's
    order of fp32 additions (_multihead.py:123-144)."""
    weighted = torch.zeros_like(neighbours[..., 0, :])
    exact_sum = torch.zeros_like(weighted)
    for r in range(neighbours.size(-2)):
        v = neighbours[..., r, :]
        weighted = weighted + v * weights[..., r].unsqueeze(-1)
        exact_sum = exact_sum + v * exact[..., r].to(neighbours.dtype).unsqueeze(-1)
    if exact.any():
        counts = exact.to(neighbours.dtype).sum(dim=-1, keepdim=True).clamp(min=1.0)
        weighted = torch.where(exact.any(dim=-1, keepdim=True), exact_sum / counts, weighted)
    return weighted


def _spread(grad: torch.Tensor, indices: torch.Tensor, weights: torch.Tensor, exact: torch.Tensor) -> torch.Tensor:
    """The transpose of `_combine` of `_gather` by tensor operations."""
    B, N, H, C = grad.shape
    hit = exact.to(grad.dtype)
    mean = grad / hit.sum(dim=-1, keepdim=True).clamp(min=1.0)
    parts = torch.where(exact.any(dim=-1, keepdim=True).unsqueeze(-1), mean.unsqueeze(-2) * hit.unsqueeze(-1),
                        grad.unsqueeze(-2) * weights.unsqueeze(-1))
    batch = torch.arange(B, device=grad.device).view(B, 1, 1, 1)
    head = torch.arange(H, device=grad.device).view(1, 1, H, 1)
    rows = ((batch * N + indices) * H + head).reshape(-1)
    zeros = torch.zeros((B * N * H, C), dtype=grad.dtype, device=grad.device)
    return zeros.index_put((rows,), parts.reshape(-1, C), accumulate=True).reshape(B, N, H, C)


class _Interpolate(torch.autograd.Function):
    """`_C.interpolate_neighbors`, differentiable (any number of times) in its
    values: the result is linear in them.  The backward may run under other
    transforms than the forward did, so it chooses again."""

    @staticmethod
    def forward(values, indices, weights, exact):
        return _C.interpolate_neighbors(values.contiguous(), indices, weights, exact)

    @staticmethod
    def setup_context(ctx, inputs, output):
        ctx.save_for_backward(*inputs[1:])

    @staticmethod
    def backward(ctx, grad):
        linear = _InterpolateTransposed.apply if _is_plain(grad) else _spread
        return linear(grad, *ctx.saved_tensors), None, None, None


class _InterpolateTransposed(torch.autograd.Function):
    """The gradient of `_Interpolate` in its values, itself linear."""

    @staticmethod
    def forward(grad, indices, weights, exact):
        return _C.interpolate_neighbors_backward(grad.contiguous(), indices, weights, exact)

    @staticmethod
    def setup_context(ctx, inputs, output):
        ctx.save_for_backward(*inputs[1:])

    @staticmethod
    def backward(ctx, grad):
        indices, weights, exact = ctx.saved_tensors
        if _is_plain(grad):
            return _Interpolate.apply(grad, indices, weights, exact), None, None, None
        return _combine(_gather(grad, indices), weights, exact), None, None, None


def _is_plain(tensor: torch.Tensor) -> bool:
    """Whether the library's kernels may take `tensor` in an autograd function:
    its memory holds its values, and no transform has to see the tensor
    operations (functorch levels, which also refuse such functions around
    tensors they don't wrap, batched gradients, forward-mode, dispatch and
    function modes, tracing)."""
    C = torch._C
    return (type(tensor) in (torch.Tensor, torch.nn.Parameter)
            and not C._are_functorch_transforms_active()
            and not C._functorch.is_legacy_batchedtensor(tensor)
            and not tensor.is_neg() and not tensor._is_zerotensor()
            and torch.autograd.forward_ad._current_level < 0
            and C._len_torch_dispatch_stack() == 0 and C._len_torch_function_stack() == 0
            and not torch.jit.is_tracing() and not torch.compiler.is_compiling())


def _kernels_differentiate(values: torch.Tensor, indices: torch.Tensor) -> bool:
    """Whether the differentiable call may run as the library's kernels: plain
    values, and entry counts the backward's sort can number."""
    return _is_plain(values) and 0 < indices.numel() <= 2**31 - 1


def interpolate_displaced(pos: torch.Tensor, q: torch.Tensor, values: torch.Tensor, k: int = 8, *,
                          reduction: str = "weighted_mean") -> torch.Tensor:
    """Inverse-squared-distance weighted mean of the matching head's values
    over the k neighbours of each displaced query, ``w = 1 / (d2 + 1e-12)``
    normalised over the neighbours; a query with exact hits (d2 <= 1e-12)
    gets the plain mean of those neighbours' values instead."""
    op = "interpolate_displaced"
    if reduction != "weighted_mean":
        raise ValueError(f"{op}: reduction must be 'weighted_mean'")
    _check_displaced(pos, q, op)
    if values.dim() != 4:
        raise ValueError(f"{op}: values must have shape (B, N, H, Ch)")
    if values.size(0) != pos.size(0) or values.size(1) != pos.size(1):
        raise ValueError(f"{op}: values first two dimensions must match pos")
    if values.size(2) != q.size(2):
        raise ValueError(f"{op}: values head dimension must match q")
    if values.size(3) < 1:
        raise ValueError(f"{op}: values must have at least one channel")
    check_cuda_f32(op, values, "values")
    if values.device != pos.device:
        raise ValueError(f"{op}: values must be on the same device as pos")
    values = dense(values)
    indices, d2 = query_displaced_knn(dense(pos), dense(q), k, return_positions=False)
    eps = EXACT_DISTANCE_EPSILON
    training = values.requires_grad and torch.is_grad_enabled()
    fused = training and _kernels_differentiate(values, indices)
    if fused:
        # Missing neighbours (index -1, always a row's last entries) are
        # refused below; the value is on its way to the host meanwhile.
        least = indices[..., -1].amin().to("cpu", non_blocking=True)
        arrived = torch.cuda.Event()
        arrived.record(torch.cuda.current_stream(indices.device))
    exact = d2 <= eps
    weights = torch.reciprocal(d2 + eps)
    weights = weights / weights.sum(dim=-1, keepdim=True).clamp(min=eps)
    if not training:
        # One kernel: the same rank-by-rank sums and exact-hit select, with
        # no gathered copy and no host synchronisation.
        return _C.interpolate_neighbors(values, indices, weights, exact)
    if fused:
        out = _Interpolate.apply(values, indices, weights, exact)
        arrived.synchronize()
        if int(least) < 0:
            raise ValueError(_NOT_LOCAL)
        return out
    return _combine(gather_neighbor_values(values, indices), weights, exact)
