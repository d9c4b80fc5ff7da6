"""The logits' gradient kernel at every width (logits per lane) and slot count
against autograd through float64 torch operators, and a layer under autocast,
whose logits have another dtype than its activations."""

from __future__ import annotations

import pytest
import torch

from astrai_amd.extension import loader, ops
from astrai_amd.model.components.autograd import RouteWeights, routing_weights
from test_gpu_backward import _random_layer


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n_tok,n_exp,top_k", [(1, 1, 1), (5, 2, 2), (130, 64, 6), (33, 65, 32), (64, 128, 8),
                                               (7, 200, 3), (9, 257, 4), (12, 1024, 32)])
def test_logits_gradient(gpu, n_tok, n_exp, top_k, dtype):
    g = torch.Generator(device=gpu).manual_seed(n_exp)
    logits = torch.randn(n_tok, n_exp, generator=g, device=gpu).to(dtype)
    dw = torch.randn(n_tok, top_k, generator=g, device=gpu).to(dtype)
    route = ops.moe_route(logits, top_k)
    got = ops.moe_route_grad(logits, route.topk_idx, dw)
    l64 = logits.double().requires_grad_(True)
    w = torch.softmax(l64, -1).gather(1, route.topk_idx.long())
    (w / w.sum(-1, keepdim=True)).backward(dw.double())
    # against exact probabilities, the kernel rounding the chosen ones v to dtype
    # (half a unit each), their sum S and the result. A logit's gradient is w_e
    # (dw_e - sum dw w), or with 0 for dw_e where e is not chosen, at most 2 w_e max
    # |dw|. In units of w_e max |dw|: S is off by 1 (its own half and the v's), so
    # the factor 1 / S by 2, the inner sum by 1.5 and its counterpart over all
    # logits by 1.5, the result's half unit 1: 6. fp32 adds its sums over the
    # logits, a few units each
    unit = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -24
    p = torch.softmax(logits.double(), -1)
    weight = p / p.gather(1, route.topk_idx.long()).sum(-1, keepdim=True)
    scale = weight * dw.double().abs().amax(-1, keepdim=True)
    err = (got.double() - l64.grad).abs() / scale
    bound = (6 if dtype == torch.bfloat16 else 40) * unit
    assert err.max().item() <= bound
    if top_k > 1:  # a gradient of zeros would not pass
        assert (l64.grad.abs() / scale).max().item() > 4 * bound


@pytest.mark.gpu
def test_layer_under_autocast_still_trains(gpu):
    layer = _random_layer(gpu, 64, 96, 4, 1, 2, torch.float32, seed=1)
    x = torch.randn(1, 40, 64, device=gpu, requires_grad=True)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        out = layer(x)
    out.sum().backward()
    assert out.dtype == torch.float32 and torch.isfinite(x.grad).all()
    assert layer.router.weight.grad is not None and torch.isfinite(layer.router.weight.grad).all()


def _route_on_cpu(logits, top_k):
    probs = torch.softmax(logits.float(), -1).to(logits.dtype)
    w, idx = probs.topk(top_k, -1)
    return ops.RouteResult(idx.int(), w / w.sum(-1, keepdim=True), torch.zeros(1, logits.shape[1], dtype=torch.int32))


def test_second_derivatives_reach_the_logits(monkeypatch):
    # create_graph: the logits' gradient is itself differentiable, as torch's operators make it
    monkeypatch.setattr(ops, "moe_route", _route_on_cpu)
    logits = torch.randn(5, 6, generator=torch.Generator().manual_seed(1), dtype=torch.float32).requires_grad_(True)
    c = torch.randn(5, 2, generator=torch.Generator().manual_seed(2))

    def second(weights):
        (g,) = torch.autograd.grad((weights * c).sum(), logits, create_graph=True)
        return g, torch.autograd.grad(g.square().sum(), logits)[0]

    topk_w, topk_idx, _ = RouteWeights.apply(logits, 2)
    got = second(topk_w)
    want = second(routing_weights(logits, topk_idx, logits.dtype))
    assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.gpu
def test_gradient_penalty_reaches_the_router(gpu):
    layer = _random_layer(gpu, 64, 96, 4, 0, 2, torch.float32, seed=1)
    x = torch.randn(1, 40, 64, device=gpu)
    (g,) = torch.autograd.grad(layer(x).square().sum(), layer.router.weight, create_graph=True)
    g.square().sum().backward()
    assert torch.isfinite(layer.router.weight.grad).all() and layer.router.weight.grad.abs().max() > 0


def test_arguments_are_checked_on_the_host():
    lib = loader.library()
    for args, word in (((16, 16, 16, 1, 10, 0, 1, 16, None), "n_experts"), ((16, 16, 16, 1, 10, 8, 9, 16, None), "top_k"),
                       ((16, 16, 16, 5, 10, 8, 2, 16, None), "dtype"), ((16, None, 16, 1, 10, 8, 2, 16, None), "null")):
        assert lib.astrai_moe_route_grad(*args) == -1 and word in loader.last_error()
    assert lib.astrai_moe_route_grad(None, None, None, 1, 0, 8, 2, None, None) == 0
