"""The autograd functions around interpolate_displaced's kernels under the
transforms that a backward may run in, on the CPU with stand-ins that, like
the kernels, take their tensors' memory: each gives what the same call by
tensor operations gives."""

import pytest
import torch
from torch.autograd import forward_ad
from torch.utils._python_dispatch import TorchDispatchMode

from torchbvh_amd import _multihead

B, N, H, C, K = 2, 7, 3, 5, 4


@pytest.fixture
def call(monkeypatch):
    """(differentiable call of `values` by the functions, the same by tensor operations)."""
    g = torch.Generator().manual_seed(1)
    indices = torch.randint(0, N, (B, N, H, K), generator=g)
    weights = torch.rand((B, N, H, K), generator=g)
    exact = torch.rand((B, N, H, K), generator=g) < 0.1

    def by_operations(values):
        out = torch.zeros_like(values)
        mean = torch.zeros_like(values)
        b, h = torch.arange(B).view(B, 1, 1), torch.arange(H).view(1, 1, H)
        for r in range(K):
            v = values[b, indices[..., r], h]
            out = out + v * weights[..., r, None]
            mean = mean + v * exact[..., r, None]
        return torch.where(exact.any(-1, keepdim=True), mean / exact.sum(-1, keepdim=True).clamp(min=1), out)

    class Kernels:
        @staticmethod
        def interpolate_neighbors(values, *rest):
            assert type(values) is torch.Tensor and not values.is_neg() and values.data_ptr() % 4 == 0
            return by_operations(values)

        @staticmethod
        def interpolate_neighbors_backward(grad, *rest):
            assert type(grad) is torch.Tensor and not grad.is_neg() and grad.data_ptr() % 4 == 0
            with torch.enable_grad():
                v = torch.zeros((B, N, H, C), requires_grad=True)
                return torch.autograd.grad(by_operations(v), v, grad)[0]

    monkeypatch.setattr(_multihead, "_C", Kernels)
    return lambda values: _multihead._Interpolate.apply(values, indices, weights, exact), by_operations


def _values(seed=2):
    return torch.randn((B, N, H, C), generator=torch.Generator().manual_seed(seed)).requires_grad_()


def _same(call, compute):
    got, want = (compute(f) for f in call)
    torch.testing.assert_close(got, want, rtol=1e-5, atol=1e-6)


def test_batched_gradients(call):
    ups = torch.randn((3, B, N, H, C))
    v = _values()
    _same(call, lambda f: torch.autograd.grad(f(v), v, ups, is_grads_batched=True)[0])


def test_vectorized_jacobian_and_its_double_backward(call):
    w = torch.randn((B, N, H, C))
    scalar = lambda f: lambda v: (f(v * v) * w).sum((1, 3))  # noqa: E731
    _same(call, lambda f: torch.autograd.functional.jacobian(scalar(f), _values(), vectorize=True))
    v, u = _values(), _values(3)

    def twice(f):
        (g,) = torch.autograd.grad(f(v), v, u, create_graph=True)
        return torch.autograd.grad(g, u, torch.stack((w, 2 * w)), is_grads_batched=True)[0]
    _same(call, twice)


def test_vmap_over_the_gradient(call):
    ups = torch.randn((3, B, N, H, C))
    v = _values()
    _same(call, lambda f: torch.func.vmap(lambda u, out=f(v): torch.autograd.grad(out, v, u, retain_graph=True)[0])(ups))


def test_gradient_with_a_tangent(call):
    up, tangent, v = torch.randn((B, N, H, C)), torch.randn((B, N, H, C)), _values()

    def compute(f):
        out = f(v)
        with forward_ad.dual_level():
            g = torch.autograd.grad(out, v, forward_ad.make_dual(up, tangent))[0]
            return tuple(forward_ad.unpack_dual(g))
    _same(call, compute)


def test_backward_under_a_dispatch_mode(call):
    class Seen(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    up, v, seen = torch.randn((B, N, H, C)), _values(), []

    def compute(f):
        out = f(v)
        with Seen():
            return torch.autograd.grad(out, v, up)[0]
    _same(call, compute)
    assert any("index_put" in str(f) for f in seen[:len(seen) // 2])


def test_negative_views(call):
    up, v = torch.randn((B, N, H, C)), _values()
    _same(call, lambda f: torch.autograd.grad(f(v), v, torch._neg_view(up))[0])


@pytest.mark.parametrize("tensor", ["plain", "neg", "function level"])
def test_the_forward_takes_the_kernels_for_plain_tensors_only(tensor):
    v = _values()
    if tensor == "function level":  # around a tensor that it does not wrap
        seen = []
        torch.func.vmap(lambda x: seen.append(_multihead._is_plain(v)) or x)(torch.zeros(2))
        assert seen == [False]
    else:
        assert _multihead._is_plain(v if tensor == "plain" else torch._neg_view(v.detach())) is (tensor == "plain")


def test_the_transpose_by_tensor_operations_in_64_bits():
    g = torch.Generator().manual_seed(5)
    idx = torch.randint(0, N, (B, N, H, K), generator=g)
    w = torch.rand((B, N, H, K), generator=g, dtype=torch.float64)
    exact = torch.rand((B, N, H, K), generator=g) < 0.2
    v = torch.randn((B, N, H, C), generator=g, dtype=torch.float64, requires_grad=True)
    up = torch.randn((B, N, H, C), generator=g, dtype=torch.float64)
    (want,) = torch.autograd.grad(_multihead._combine(_multihead._gather(v, idx), w, exact), v, up)
    torch.testing.assert_close(_multihead._spread(up, idx, w, exact), want, rtol=1e-14, atol=1e-14)
