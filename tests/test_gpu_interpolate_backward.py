"""The values' gradient of interpolate_displaced by the library's kernels
(csrc/interp.hip) against the same call by tensor operations and against 64
bits, over channel layouts, key ranges of one to three sort digits, exact
hits, strided values and gradients, and the autograd features that go through
it or round it."""

import pytest
import torch

import torchbvh_amd as tb
from torchbvh_amd import _multihead
from torchbvh_amd._native import _C

pytestmark = pytest.mark.gpu


def _inputs(B, N, H, D, C, seed):
    g = torch.Generator("cuda").manual_seed(seed)
    pos = torch.rand((B, N, D), generator=g, device="cuda")
    pos[:, : N // 4] = pos[:, N // 4 : 2 * (N // 4)]  # exact hits of two points
    q = pos[:, :, None, :] + 0.02 * torch.randn((B, N, H, D), generator=g, device="cuda")
    q[:, ::3, 0] = pos[:, ::3]
    values = torch.randn((B, N, H, C), generator=g, device="cuda")
    up = torch.randn((B, N, H, C), generator=g, device="cuda")
    return pos, q.contiguous(), values, up


def _grad(pos, q, values, up, k):
    v = values.detach().requires_grad_()
    out = tb.interpolate_displaced(pos, q, v, k)
    (g,) = torch.autograd.grad(out, v, up)
    return out.detach(), g


@pytest.mark.parametrize("B,N,H,D,C,k", [(1, 40, 1, 3, 4, 4), (2, 127, 2, 2, 1, 8), (1, 300, 3, 3, 13, 16),
                                         (3, 1031, 4, 3, 16, 8), (2, 700, 1, 2, 33, 32), (1, 20_001, 4, 3, 8, 4)])
def test_kernels_match_tensor_operations(monkeypatch, B, N, H, D, C, k):
    pos, q, values, up = _inputs(B, N, H, D, C, N + C)
    out, grad = _grad(pos, q, values, up, k)
    assert torch.equal(grad, _grad(pos, q, values, up, k)[1])  # one order of sums
    monkeypatch.setattr(_multihead, "_kernels_differentiate", lambda *a: False)
    want_out, want = _grad(pos, q, values, up, k)
    assert torch.equal(out, want_out)
    # 64-bit sums from the same coefficients; every term has two roundings and
    # a sum of m terms m more: (m + 2) eps of the sum of magnitudes.
    idx, d2 = tb.query_displaced_knn(pos, q, k, return_positions=False)
    hit = d2 <= 1e-12
    w = torch.reciprocal(d2 + 1e-12)
    w = (w / w.sum(-1, keepdim=True).clamp(min=1e-12)).double()
    w = torch.where(hit.any(-1, keepdim=True), hit / hit.double().sum(-1, keepdim=True).clamp(min=1.0), w)
    exact, size, terms = (torch.zeros(values.shape, dtype=torch.float64, device="cuda") for _ in range(3))
    b = torch.arange(B, device="cuda").view(B, 1, 1).expand(B, N, H)
    h = torch.arange(H, device="cuda").view(1, 1, H).expand(B, N, H)
    for r in range(k):
        term = w[..., r, None] * up.double()
        exact.index_put_((b, idx[..., r], h), term, accumulate=True)
        size.index_put_((b, idx[..., r], h), term.abs(), accumulate=True)
        terms.index_put_((b, idx[..., r], h), torch.ones_like(term), accumulate=True)
    bound = (terms + 2) * 2.0**-23 * size
    assert ((grad.double() - exact).abs() <= bound).all()
    assert ((want.double() - exact).abs() <= bound).all()


def test_strided_values_and_gradients():
    pos, q, values, up = _inputs(2, 200, 3, 3, 8, 1)
    _, want = _grad(pos, q, values, up, 8)
    wide = torch.randn((2, 3, 200, 8), device="cuda")
    wide.copy_(values.transpose(1, 2))
    v = wide.transpose(1, 2).requires_grad_()
    out = tb.interpolate_displaced(pos, q, v, 8)
    (g,) = torch.autograd.grad(out, v, up.transpose(0, 3).contiguous().transpose(0, 3))
    assert torch.equal(g, want)
    v = values.clone().requires_grad_()
    tb.interpolate_displaced(pos, q, v, 8).sum().backward()  # an expanded gradient
    assert torch.equal(v.grad, _grad(pos, q, values, torch.ones_like(up), 8)[1])


def test_differentiates_again_forward_mode_and_saved_tensor_hooks():
    pos, q, values, up = _inputs(1, 64, 2, 3, 3, 2)
    _, grad = _grad(pos, q, values, up, 4)
    # Linear: the gradient of <grad(u), c> in u is the forward of c.
    v = values.clone().requires_grad_()
    u = up.clone().requires_grad_()
    (g,) = torch.autograd.grad(tb.interpolate_displaced(pos, q, v, 4), v, u, create_graph=True)
    c = torch.randn_like(g)
    (gg,) = torch.autograd.grad(g, u, c)
    assert torch.equal(gg, _grad(pos, q, c, up, 4)[0])
    f = lambda x: tb.interpolate_displaced(pos, q, x, 4)  # noqa: E731
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(values.clone().requires_grad_(), c)
        tangent = torch.autograd.forward_ad.unpack_dual(f(dual)).tangent
    torch.testing.assert_close(tangent, _grad(pos, q, c, up, 4)[0], rtol=1e-6, atol=1e-6)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), lambda t: t.cuda()):
        assert torch.equal(_grad(pos, q, values, up, 4)[1], grad)


def test_missing_neighbours_are_refused():
    pos, q, values, _ = _inputs(1, 40, 1, 3, 4, 3)
    q[0, 5] = float("inf")
    with pytest.raises(ValueError, match="indices must be local source indices"):
        tb.interpolate_displaced(pos, q, values.requires_grad_(), 4)


def test_binding_indices_out_of_range_add_nothing():
    g = torch.Generator("cuda").manual_seed(4)
    idx = torch.randint(-3, 13, (2, 10, 2, 4), generator=g, device="cuda")
    w = torch.rand((2, 10, 2, 4), generator=g, device="cuda")
    up = torch.randn((2, 10, 2, 5), generator=g, device="cuda")
    none = torch.zeros_like(w, dtype=torch.bool)
    got = _C.interpolate_neighbors_backward(up, idx, w, none)
    valid = (idx >= 0) & (idx < 10)
    assert torch.equal(got, _C.interpolate_neighbors_backward(up, idx.clamp(0, 9), w * valid, none))


@pytest.mark.parametrize("how", ["batched", "vmap", "tangent", "around"])
def test_backward_under_transforms(monkeypatch, how):
    """The forward ran in the kernels; the backward meets transforms that they
    can't take (and the forward itself, one around plain values)."""
    pos, q, values, up = _inputs(1, 64, 2, 3, 3, 6)
    ups = torch.randn((3, *up.shape), generator=torch.Generator("cuda").manual_seed(7), device="cuda")

    def compute():
        v = values.clone().requires_grad_()
        if how == "around":
            f = lambda s: (s * tb.interpolate_displaced(pos, q, v, 4) * up).sum()  # noqa: E731
            return torch.autograd.grad(torch.func.vmap(f)(torch.ones(2, device="cuda")).sum(), v)[0]
        out = tb.interpolate_displaced(pos, q, v, 4)
        if how == "batched":
            return torch.autograd.grad(out, v, ups, is_grads_batched=True)[0]
        if how == "vmap":
            return torch.func.vmap(lambda u: torch.autograd.grad(out, v, u, retain_graph=True)[0])(ups)
        with torch.autograd.forward_ad.dual_level():
            g = torch.autograd.grad(out, v, torch.autograd.forward_ad.make_dual(ups[0], ups[1]))[0]
            return torch.stack(tuple(torch.autograd.forward_ad.unpack_dual(g)))

    got = compute()
    monkeypatch.setattr(_multihead, "_kernels_differentiate", lambda *a: False)
    # Sums of up to 64 terms of size about one, in another order.
    torch.testing.assert_close(got, compute(), rtol=0, atol=64 * 2.0**-22)
