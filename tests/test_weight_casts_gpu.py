"""The linear layers' parameters cast by one launch per block: the bits that autocast's own casts give, in every mode that reaches
the layers, and none of it where a layer is more than its class."""
import pytest
import torch

from semicat_amd import adaln, train_step
from semicat_amd.dit import DIT, _linear

pytestmark = pytest.mark.gpu


def _net():
    torch.manual_seed(0)
    net = DIT(48, 128, 16, 2, 2, 0.0, 16).cuda()
    for p in net.parameters():
        if not p.any():
            torch.nn.init.normal_(p, std=0.05)
    return net, torch.randn(4, 16, 48, device="cuda"), torch.randint(0, 48, (4, 16), device="cuda")


def _step(net, x0, x1, create_graph=False):
    t = torch.linspace(0.2, 0.8, 4, device="cuda")
    with torch.autocast("cuda", dtype=torch.bfloat16):
        vf = train_step.vfm_loss(net, x0[2:], x1[2:], t=t[2:])
        sd = train_step.lag_self_distillation_loss(net, x0[:2], x1[:2], t=t[:2], s=t[:2] / 2)
    loss = vf if create_graph else vf + sd  # (the op itself cannot be differentiated twice)
    return [vf, sd, *torch.autograd.grad(loss, list(net.parameters()), create_graph=create_graph)]


def test_same_bits_as_autocast(monkeypatch):
    net, x0, x1 = _net()
    served = []
    cast = adaln.cast
    monkeypatch.setattr(adaln, "cast", lambda *m: served.append(cast(*m)) or served[-1])
    got = _step(net, x0, x1)
    assert len(served) == 3 * 3 and all(c is not None for c in served)
    monkeypatch.setattr(adaln, "cast", lambda *m: None)
    for a, b in zip(got, _step(net, x0, x1)):
        assert a.dtype == b.dtype and a.stride() == b.stride() and torch.equal(a, b)


def test_frozen_parameters_and_no_grad(monkeypatch):
    net, x0, x1 = _net()
    net.blocks[0].attn_qkv.weight.requires_grad_(False)
    net.blocks[1].mlp[0].bias.requires_grad_(False)

    def run():
        net.zero_grad(set_to_none=True)
        with torch.autocast("cuda", dtype=torch.bfloat16):
            loss = train_step.vfm_loss(net, x0, x1, t=torch.full((4,), 0.5, device="cuda"))
            with torch.no_grad():
                out = net(x0, *torch.full((2, 4), 0.25, device="cuda"))
        loss.backward()
        return [loss, out, *(p.grad for p in net.parameters())]

    got = run()
    monkeypatch.setattr(adaln, "cast", lambda *m: None)
    for a, b in zip(got, run()):
        assert (a is None) == (b is None) and (a is None or torch.equal(a, b))


def test_copies_of_plain_calls():
    """A node for each parameter that needs one; gradients reach the layers one after the other."""
    layers = [torch.nn.Linear(24, 40, device="cuda"), torch.nn.Linear(40, 16, device="cuda")]
    layers[0].weight.requires_grad_(False)
    order = []
    for i, m in enumerate(layers):
        m.bias.register_post_accumulate_grad_hook(lambda p, i=i: order.append(i))
    copies = adaln.cast(*layers)
    for m in layers:
        for p, c in zip((m.weight, m.bias), copies[m]):
            assert c.dtype == torch.bfloat16 and c.requires_grad == p.requires_grad and torch.equal(c, p.bfloat16())
    z = adaln.plain_linear(layers[0], torch.randn(3, 24, device="cuda").bfloat16(), copies)
    z.register_hook(lambda g: order.append("between"))
    y = adaln.plain_linear(layers[1], z, copies)
    only, = torch.autograd.grad(y.sum(), layers[1].bias, retain_graph=True)
    assert order == [] and only.dtype == torch.float32
    y.sum().backward()
    assert order.index(1) < order.index(0) and layers[0].weight.grad is None and torch.equal(layers[1].bias.grad, only)
    with torch.no_grad():
        assert not any(c.requires_grad for c in adaln.cast(*layers)[layers[1]])


@pytest.mark.parametrize("mode", [torch.no_grad, torch.inference_mode])
def test_calls_in_one_autocast_region(mode):
    """A call without gradients leaves the ones behind it theirs; two that record add theirs up in float32."""
    layer = torch.nn.Linear(24, 40, device="cuda")
    x = torch.randn(3, 24, device="cuda").bfloat16()
    with torch.autocast("cuda", dtype=torch.bfloat16):
        with mode():
            y = _linear(True, layer, x, adaln.cast(layer))
        ys = [adaln.plain_linear(layer, x * scale, adaln.cast(layer)) for scale in (1.0, 2 ** -9)]
    assert not y.requires_grad and torch.equal(y, ys[0])
    grads = [torch.autograd.grad(z.sum(), layer.weight, retain_graph=True)[0] for z in ys]
    (ys[0].sum() + ys[1].sum()).backward()
    assert torch.equal(layer.weight.grad, grads[0] + grads[1])


def test_region_without_gradients(monkeypatch):
    """Calls of the network in one region cast its parameters once, frozen ones excepted; the bits are autocast's own."""
    net, x0, _ = _net()
    net.blocks[0].attn_qkv.weight.requires_grad_(False)
    t = torch.full((4,), 0.25, device="cuda")
    made = []
    cast_all = adaln.functional._cast_all
    monkeypatch.setattr(adaln.functional, "_cast_all", lambda ts, ds: made.append(sum(z is not None for z in ts)) or cast_all(ts, ds))

    def run(**region):
        with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16, **region):
            return [net(x0, t, t), net(x0, t, t)]

    got = run()
    assert made == [1, 1]
    got += run(cache_enabled=False)
    assert made[2:] == [8, 8, 4] * 2
    monkeypatch.setattr(adaln, "cast", lambda *m: None)
    want = run()[0]
    assert all(torch.equal(y, want) for y in got)


def test_recorded_backward(monkeypatch):
    """Gradients that are recorded, of the network's plain call and of a dual layer, and the gradients of those."""
    net, x0, x1 = _net()
    got = _step(net, x0, x1, create_graph=True)
    cast = adaln.cast
    monkeypatch.setattr(adaln, "cast", lambda *m: None)
    for a, b in zip(got, _step(net, x0, x1, create_graph=True)):
        assert a.dtype == b.dtype and torch.equal(a, b)
    monkeypatch.setattr(adaln, "cast", cast)
    layer = torch.nn.Linear(24, 40, device="cuda")

    def twice(copies):
        torch.manual_seed(1)
        x, t = (torch.randn(6, 24, device="cuda").bfloat16().requires_grad_() for _ in range(2))
        out = torch.func.jvp(lambda z: adaln.linear(layer, z, adaln.cast(layer) if copies else None), (x,), (t,))
        first = torch.autograd.grad(out, [x, t, layer.weight, layer.bias], [torch.ones_like(z) for z in out], create_graph=True)
        return [*out, *first, *torch.autograd.grad(sum(g.float().pow(2).sum() for g in first), [x, t, layer.weight])]

    for a, b in zip(twice(True), twice(False)):
        assert a.dtype == b.dtype and torch.equal(a, b)


def test_layers_that_are_left_to_pytorch():
    net, _, _ = _net()
    block = net.blocks[0]
    assert adaln.cast(block.attn_qkv, block.attn_out) is not None
    handle = block.attn_out.register_forward_hook(lambda *a: None)
    assert adaln.cast(block.attn_qkv, block.attn_out) is None
    handle.remove()
    assert adaln.cast(block.attn_qkv, torch.nn.Linear(4, 4)) is None  # another device
    assert adaln.cast(torch.nn.Linear(4, 4, device="cuda", dtype=torch.bfloat16)) is None
    assert adaln.cast(torch.nn.utils.parametrizations.weight_norm(torch.nn.Linear(4, 4, device="cuda"))) is None
    with torch.autograd.forward_ad.dual_level():
        assert adaln.cast(block.attn_qkv) is None
    torch.func.vmap(lambda z: (adaln.cast(block.attn_qkv) is None or 1 / 0, z)[1])(torch.zeros(2, device="cuda"))
    torch.func.grad(lambda z: (adaln.cast(block.attn_qkv) is None or 1 / 0, z)[1])(torch.zeros((), device="cuda"))
