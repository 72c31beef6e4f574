"""The copies that a block's linear layers share are values: a layer's parameters keep their own places in the graph.  (CPU; the
cast itself is PyTorch's here.)"""
import torch
from torch import nn

from semicat_amd import adaln


def _layers(monkeypatch):
    monkeypatch.setattr(torch.Tensor, "is_cuda", True, raising=False)
    torch.manual_seed(0)
    return nn.Linear(24, 40), nn.Linear(40, 16), nn.Linear(16, 8, bias=False)


def _dual(layers, copies=True):
    """The layers one behind the other on a dual tensor, with shared copies or each for itself."""
    x, t = (torch.randn(6, 24).bfloat16().requires_grad_() for _ in range(2))

    def run(z):
        shared = adaln.cast(*layers) if copies else None
        for m in layers:
            z = adaln.linear(m, z, shared)
        return z

    return torch.func.jvp(run, (x,), (t,))


def test_copies_of_frozen_parameters_cost_no_gradient(monkeypatch):
    layers = _layers(monkeypatch)
    products = []
    mm = torch.mm

    def backward():
        out = _dual(layers)
        monkeypatch.setattr(torch, "mm", lambda *a, **k: products.append(1) or mm(*a, **k))
        torch.autograd.backward(out, [torch.ones_like(z) for z in out])
        monkeypatch.setattr(torch, "mm", mm)
        return len(products), products.clear()

    everything, _ = backward()
    assert everything == 6 and all(p.grad is not None for m in layers for p in m.parameters())
    for m in layers:
        m.weight.grad = None
    layers[0].weight.requires_grad_(False)
    layers[2].weight.requires_grad_(False)
    assert backward()[0] == everything - 2 and layers[0].weight.grad is None and layers[1].weight.grad is not None


def test_one_gradient_asked_for_takes_one_layers_backward(monkeypatch):
    layers = _layers(monkeypatch)
    out = _dual(layers)
    products = []
    mm = torch.mm
    monkeypatch.setattr(torch, "mm", lambda *a, **k: products.append(1) or mm(*a, **k))
    torch.autograd.grad(out, layers[2].weight, [torch.ones_like(z) for z in out])
    assert len(products) == 2  # of the input and of the weight


def test_gradients_arrive_layer_by_layer(monkeypatch):
    """What waits for a parameter's gradient (an optimizer in the backward, a bucket of a reduction) starts while the
    layers in front of it are still to come."""
    layers = _layers(monkeypatch)
    order = []
    for i, m in enumerate(layers):
        m.weight.register_post_accumulate_grad_hook(lambda p, i=i: order.append(("gradient", i)))
    shape = {m.weight.shape: i for i, m in enumerate(layers)}
    backward = adaln.LinearFunction.backward

    def noted(ctx, *g):
        order.append(("backward", shape[ctx.saved_tensors[2].shape]))
        return backward(ctx, *g)

    monkeypatch.setattr(adaln.LinearFunction, "backward", staticmethod(noted))
    out = _dual(layers)
    torch.autograd.backward(out, [torch.ones_like(z) for z in out])
    assert order == [(what, i) for i in (2, 1, 0) for what in ("backward", "gradient")]


def test_copies_give_what_each_layers_own_cast_gives(monkeypatch):
    layers = _layers(monkeypatch)
    res = []
    for copies in (True, False):
        torch.manual_seed(1)
        out = _dual(layers, copies)
        res.append([*out, *torch.autograd.grad(out, [p for m in layers for p in m.parameters()], [torch.ones_like(z) for z in out])])
    for a, b in zip(*res):
        assert a.dtype == b.dtype and torch.equal(a, b)


def test_calls_without_gradients_share_the_regions_casts(monkeypatch):
    """What autocast keeps for a region is not cast once more for each call in it; what it does not keep still is."""
    layers = _layers(monkeypatch)
    monkeypatch.setattr(torch, "is_autocast_enabled", lambda *device: True)
    with torch.no_grad():
        assert torch.is_autocast_cache_enabled() and adaln.cast(*layers) is None
        assert adaln.cast(layers[0], nn.Sequential(layers[1])) is None  # no weight of its own
        layers[1].weight.requires_grad_(False)
        copies = adaln.cast(*layers)
        own = [c is not p for m in layers for p, c in zip((m.weight, m.bias), copies[m]) if p is not None]
        assert own == [False, False, True, False, False] and torch.equal(copies[layers[1]][0], layers[1].weight.bfloat16())
        torch.set_autocast_cache_enabled(False)
        try:
            copies = adaln.cast(*layers)
        finally:
            torch.set_autocast_cache_enabled(True)
    assert all(c is None or c.dtype == torch.bfloat16 for pair in copies.values() for c in pair)
    for m in layers:
        m.requires_grad_(False)
    assert all(c is None or c.dtype == torch.bfloat16 for pair in adaln.cast(*layers).values() for c in pair)
