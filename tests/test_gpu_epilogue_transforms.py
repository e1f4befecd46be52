"""Backward of the fused bias + ReLU under what torch may do to the tensors it hands over: saved-tensor
hooks, batched and dual upstream gradients, lazy negation, recorded backward passes.  Only the bias
requires a gradient, so that nothing but the epilogue's gradient runs."""
import pytest
import torch
from torch.autograd import forward_ad
from torch.fx.experimental.proxy_tensor import make_fx

from approxtrain_amd.layers import AMConv2D
from tests.util import lut_path

pytestmark = pytest.mark.gpu


def _layer(hooks=None):
    gen = torch.Generator(device="cuda").manual_seed(5)
    layer = AMConv2D(6, 3, activation="relu", mant_mul_lut=lut_path("MBM", 5), in_channels=3).cuda()
    layer.kernel.requires_grad_(False)
    x = torch.randn((2, 8, 9, 3), device="cuda", generator=gen)
    if hooks is None:
        out = layer(x)
    else:
        with torch.autograd.graph.saved_tensors_hooks(*hooks):
            out = layer(x)
    return layer, out, torch.randn(out.shape, device="cuda", generator=gen)


def _want(out, dy):
    return (dy * (out.detach() > 0)).reshape(-1, dy.shape[-1]).sum(0)


def _close(got, want):
    # 84 terms below 64 (dy * dy at four deviations and more), added in another order
    assert torch.allclose(got, want, rtol=0, atol=84 * 2.0 ** -24 * 84 * 64)


def test_saved_output_in_another_type():
    def pack(t):
        return t.half() if t.shape == (2, 6, 7, 6) else t
    layer, out, dy = _layer((pack, lambda t: t))
    (gb,) = torch.autograd.grad(out, layer.bias, dy)
    _close(gb, _want(out.half(), dy))


def test_batched_upstream_gradients():
    layer, out, dy = _layer()
    dys = torch.stack((dy, -2.0 * dy, dy * dy))
    (gb,) = torch.autograd.grad(out, layer.bias, dys, is_grads_batched=True)
    for got, d in zip(gb, dys):
        _close(got, _want(out, d))


def test_dual_upstream_gradient_keeps_its_tangent():
    layer, out, dy = _layer()
    tangent = dy.flip(0)
    with forward_ad.dual_level():
        (gb,) = torch.autograd.grad(out, layer.bias, forward_ad.make_dual(dy, tangent))
        primal, got = forward_ad.unpack_dual(gb)
        assert got is not None
        _close(primal, _want(out, dy))
        _close(got, _want(out, tangent))


def test_lazily_negated_upstream_gradient():
    layer, out, dy = _layer()
    (gb,) = torch.autograd.grad(out, layer.bias, torch._neg_view(dy))
    _close(gb, -_want(out, dy))


def test_recorded_backward_pass_serves_other_gradients():
    layer, out, dy = _layer()
    recorded = make_fx(lambda d: torch.autograd.grad(out, layer.bias, d, retain_graph=True)[0])(dy)
    other = dy.flip(0) * 3.0
    _close(recorded(other), _want(out, other))


def test_efficient_zero_upstream_gradient():
    layer, out, dy = _layer()
    (gb,) = torch.autograd.grad(out, layer.bias, torch._efficientzerotensor(dy.shape, device="cuda"))
    assert torch.equal(gb + torch.zeros_like(layer.bias), torch.zeros_like(layer.bias))
