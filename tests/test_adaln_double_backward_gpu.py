"""Backwards that are differentiated again: the fused functions of the DiT's blocks as PyTorch's operations served them, the
attention op with its own refusal."""
import pytest
import torch
import torch.nn.functional as F

from semicat_amd import adaln, train_step
from semicat_amd.dit import DIT
from tests.test_adaln_convention import _written_out

pytestmark = pytest.mark.gpu
# First and second gradients pass through bf16 two to four times: 2^-9 each.
TOL = 2e-2


def _rand(gen, *shape, dtype=torch.bfloat16, scale=1.0):
    return (torch.randn(shape, generator=gen, device="cuda") * scale).to(dtype).requires_grad_()


def _second(outs, inputs, cots, weights):
    """Gradients, and the gradients of a weighted sum of them, with respect to the inputs and the cotangents."""
    first = torch.autograd.grad(outs, inputs, cots, create_graph=True)
    total = sum((g * w).sum() for g, w in zip(first, weights))
    return first, torch.autograd.grad(total, (*inputs, *cots), allow_unused=True)


def _compare(outs, inputs, reference, cots):
    gen = torch.Generator("cuda").manual_seed(7)
    weights = [torch.randn(z.shape, generator=gen, device="cuda") for z in inputs]
    got = _second(outs, inputs, cots, weights)
    d = [z.detach().double().requires_grad_() for z in inputs]
    dc = [c.detach().double().requires_grad_() for c in cots]
    ref = _second(reference(*d), d, dc, [w.double() for w in weights])
    for order in (0, 1):
        for i, (a, r) in enumerate(zip(got[order], ref[order])):
            assert (a is None) == (r is None) or r is None or not r.any(), (order, i)
            if a is not None and r is not None:
                assert (a.double() - r).norm() <= TOL * r.norm() + 1e-6, (order, i)


@pytest.mark.parametrize("mode", ["gate", "norm", "both"])
@pytest.mark.parametrize("jvp", [False, True])
@pytest.mark.parametrize("strided", [False, True])
def test_gated_norm(mode, jvp, strided):
    B, S, W = 3, 5, 64
    gen = torch.Generator("cuda").manual_seed(1)
    gate, norm = mode != "norm", mode != "gate"
    act = lambda: (_rand(gen, B, S, 2 * W)[..., ::2].detach().requires_grad_() if strided else _rand(gen, B, S, W))
    names = {"x": act()}
    if gate:
        names.update(a=act(), gate=_rand(gen, B, 1, W))
    if norm:
        names.update(scale=_rand(gen, B, 1, W, scale=0.5), shift=_rand(gen, B, 1, W), w=_rand(gen, W, dtype=torch.float32),
                     b=_rand(gen, W, dtype=torch.float32))
    if jvp:
        names["tx"] = act()
        if gate:
            names.update(ta=act(), tgate=_rand(gen, B, 1, W))
        if norm:
            names.update(tscale=_rand(gen, B, 1, W), tshift=_rand(gen, B, 1, W))
    t = {n: names.get(n) for n in adaln._ARGUMENTS}
    y, h, ty, th = adaln.GatedNormFunction.apply(1e-5, jvp, *t.values())
    outs = [z for z in (y, h, ty, th) if z is not None]

    def reference(*values):
        v = dict(dict.fromkeys(adaln._ARGUMENTS), **dict(zip(names, values)))
        y, ty = v["x"], v["tx"]
        res = []
        if gate:
            y = v["a"] * v["gate"] + y
            ty = v["ta"] * v["gate"] + v["a"] * v["tgate"] + ty if jvp else None
            res += [y]
        if norm:
            zero = torch.zeros_like(y)
            h, th = _written_out(y, ty if jvp else zero, v["w"], v["b"], v["scale"], v["tscale"] if jvp else 0.0 * v["scale"],
                                 v["shift"], v["tshift"] if jvp else 0.0 * v["shift"], 1e-5)
            res += [h]
        if jvp:
            res += ([ty] if gate else []) + ([th] if norm else [])
        return res

    cots = [torch.randn(B, S, W, generator=gen, device="cuda").bfloat16().requires_grad_() for _ in outs]
    _compare(outs, tuple(names.values()), reference, cots)


@pytest.mark.parametrize("jvp", [False, True])
def test_gelu(jvp):
    gen = torch.Generator("cuda").manual_seed(2)
    x = (_rand(gen, 512, scale=2.0), _rand(gen, 512)) if jvp else (_rand(gen, 512, scale=2.0),)
    outs = [z for z in adaln.GeluFunction.apply(x[0], x[1] if jvp else None) if z is not None]

    def reference(u, tu=None):
        y = F.gelu(u, approximate="tanh")
        return [y] if tu is None else [y, torch.autograd.grad(y.sum(), u, create_graph=True)[0] * tu]

    _compare(outs, x, reference, [_rand(gen, 512) for _ in outs])


@pytest.mark.parametrize("bias", [False, True])
def test_linear_with_weights_that_have_changed_since(bias):
    gen = torch.Generator("cuda").manual_seed(3)
    x = [_rand(gen, 4, 6, 24), _rand(gen, 4, 6, 24), _rand(gen, 40, 24).detach().float().requires_grad_()]
    if bias:
        x.append(_rand(gen, 40, dtype=torch.float32))
    outs = adaln.LinearFunction.apply(*x, *(() if bias else (None,)))
    cots = [_rand(gen, 4, 6, 40) for _ in outs]
    ref = lambda x, tx, w, b=None: (F.linear(x, w, b), F.linear(tx, w))
    _compare(outs, x, ref, cots)
    first = torch.autograd.grad(outs, x[:2], cots, retain_graph=True)
    with torch.no_grad():
        x[2].zero_()  # an optimizer's step: the layer keeps the values that it computed with
    for a, r in zip(torch.autograd.grad(outs, x[:2], cots, create_graph=True), first):
        assert torch.equal(a, r)


def _network_and_data():
    torch.manual_seed(0)
    net = DIT(48, 128, 16, 2, 2, 0.0, 16).cuda()
    for p in net.parameters():
        if not p.any():
            torch.nn.init.normal_(p, std=0.05)
    t = torch.rand(4, device="cuda") * 0.5 + 0.4
    return net, torch.randn(4, 16, 48, device="cuda"), torch.randint(0, 48, (4, 16), device="cuda"), t


@pytest.mark.parametrize("name", ["output_layer.linear.weight", "output_layer.norm_final.weight"])
@pytest.mark.parametrize("jvp", [False, True])
def test_last_layers_of_the_network(monkeypatch, name, jvp):
    """A penalty on the gradient of parameters behind the last attention: nothing of the op is differentiated twice."""
    def run():
        net, x0, x1, t = _network_and_data()
        with torch.autocast("cuda", dtype=torch.bfloat16):
            loss = train_step.lag_self_distillation_loss(net, x0, x1, t=t, s=t * 0.5) if jvp \
                else net(x0, t, t).float().pow(2).mean()
        p = net.get_parameter(name)
        g, = torch.autograd.grad(loss, p, create_graph=True)
        g.pow(2).sum().backward()
        return p.grad

    got = run()
    monkeypatch.setattr(adaln, "serves_block", lambda x: False)
    ref = run()
    assert (got - ref).norm() < 5e-2 * ref.norm()


@pytest.mark.parametrize("jvp", [False, True])
def test_the_op_refuses(jvp):
    net, x0, x1, t = _network_and_data()
    with torch.autocast("cuda", dtype=torch.bfloat16):
        loss = train_step.lag_self_distillation_loss(net, x0, x1, t=t, s=t * 0.5) if jvp \
            else train_step.vfm_loss(net, x0, x1, t=t)
    grads = torch.autograd.grad(loss, list(net.parameters()), create_graph=True)
    with pytest.raises(NotImplementedError, match="double backward"):
        sum(g.pow(2).sum() for g in grads).backward()
