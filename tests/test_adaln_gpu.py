"""The fused element-wise kernels of the DiT's blocks (csrc/sjvp_adaln.hip) against the PyTorch operations in fp64.
(PyTorch's reverse mode of a forward-mode layer_norm holds the statistics of its input constant; the kernels give the
same gradients.)"""
import pytest
import torch
import torch.nn.functional as F

from semicat_amd import adaln, train_step
from semicat_amd.dit import DIT

pytestmark = pytest.mark.gpu

# A result is rounded to bf16 once (relative 2^-9 at most, 2^-9 / sqrt(3) in the root mean square); with a gate the norm
# reads y behind its own rounding, which adds another such error in y and, through it, in everything behind: below 1e-2.
TOL = 1e-2


def _check(name, got, ref):
    err = (got.double() - ref).norm() / ref.norm().clamp_min(1e-30)
    assert err < TOL, f"{name}: {err:.2e}"


def _reference(eps, jvp, x, a, gate, scale, shift, w, b, tx, ta, tgate, tscale, tshift):
    def f(x, a, gate, scale, shift):
        y = x if a is None else a * gate + x
        return y, y if w is None else F.layer_norm(y, w.shape, w, b, eps) * (1 + scale) + shift

    primals = (x, a, gate, scale, shift)
    if not jvp:
        return (*f(*primals), None, None)
    at = [i for i, p in enumerate(primals) if p is not None]

    def g(*some):
        full = list(primals)
        for i, p in zip(at, some):
            full[i] = p
        return f(*full)

    tangents = (tx, ta, tgate, tscale, tshift)
    (y, h), (ty, th) = torch.func.jvp(g, tuple(primals[i] for i in at), tuple(
        torch.zeros_like(primals[i]) if tangents[i] is None else tangents[i] for i in at))
    return y, h, ty, th


@pytest.mark.parametrize("mode", ["gate", "norm", "both"])
@pytest.mark.parametrize("jvp", [False, True])
@pytest.mark.parametrize("B,S,W", [(1, 1, 8), (3, 17, 256), (2, 33, 264), (16, 128, 768), (5, 9, 1024)])
def test_gated_norm_against_fp64(mode, jvp, B, S, W):
    gen = torch.Generator("cuda").manual_seed(B * W + S)

    def rand(*shape, dtype=torch.bfloat16, scale=1.0):
        return (torch.randn(shape, generator=gen, device="cuda") * scale).to(dtype).requires_grad_()

    gate, norm = mode != "norm", mode != "gate"
    modulation = rand(B, 6 * W, scale=0.5).detach()[:, None].chunk(6, dim=2)  # rows of a wider projection
    mods = [m.requires_grad_() for m in modulation]
    t = [rand(B, S, W), rand(B, S, W) if gate else None, mods[0] if gate else None, mods[1] if norm else None,
         mods[2] if norm else None, rand(W, dtype=torch.float32) if norm else None,
         rand(W, dtype=torch.float32) if norm else None]
    t += [rand(B, S, W), rand(B, S, W) if gate else None, mods[3] if gate else None, mods[4] if norm else None,
          mods[5] if norm else None] if jvp else [None] * 5
    if jvp and mode == "norm":
        t[7] = None  # the first block: only the modulation has a tangent
    outs = adaln.GatedNormFunction.apply(1e-5, jvp, *t)
    ref_in = [None if p is None else p.detach().double().requires_grad_() for p in t]
    refs = _reference(1e-5, jvp, *ref_in)
    keep = [i for i in range(4) if outs[i] is not None]
    assert keep == [i for i, on in enumerate((gate, norm, gate and jvp, norm and jvp)) if on]
    cot = {i: torch.randn(B, S, W, generator=gen, device="cuda").bfloat16() for i in keep}
    for i in keep:
        _check(f"output {i}", outs[i], refs[i])
    wrt = [i for i, p in enumerate(t) if p is not None]
    got = torch.autograd.grad([outs[i] for i in keep], [t[i] for i in wrt], [cot[i] for i in keep])
    ref = torch.autograd.grad([refs[i] for i in keep], [ref_in[i] for i in wrt], [cot[i].double() for i in keep],
                              allow_unused=True)
    for i, g, r in zip(wrt, got, ref):
        assert g.shape == t[i].shape and g.dtype == t[i].dtype
        _check(f"gradient {i}", g, torch.zeros_like(ref_in[i]) if r is None else r)


@pytest.mark.parametrize("n", [8, 2056, 1 << 18])
def test_gelu_against_fp64(n):
    gen = torch.Generator("cuda").manual_seed(n)
    u, tu, dy, dty = ((torch.randn(n, generator=gen, device="cuda") * s).bfloat16() for s in (3.0, 1.0, 1.0, 1.0))
    u.requires_grad_(), tu.requires_grad_()
    outs = adaln.GeluFunction.apply(u, tu)
    u64, tu64 = (z.detach().double().requires_grad_() for z in (u, tu))
    refs = torch.func.jvp(lambda z: F.gelu(z, approximate="tanh"), (u64,), (tu64,))
    for name, got, ref in zip(("y", "ty", "du", "dtu"), (*outs, *torch.autograd.grad(outs, (u, tu), (dy, dty))),
                              (*refs, *torch.autograd.grad(refs, (u64, tu64), (dy.double(), dty.double())))):
        _check(name, got, ref)


@pytest.mark.parametrize("adjacent", [False, True])
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("cot", ["both", "y", "ty"])
def test_linear_against_fp64(adjacent, bias, cot):
    gen = torch.Generator("cuda").manual_seed(3)
    x, tx = torch.randn(2, 3, 5, 24, generator=gen, device="cuda").bfloat16().unbind(0)
    if not adjacent:
        tx = tx.clone()
    x.requires_grad_(), tx.requires_grad_()
    w = torch.randn(40, 24, generator=gen, device="cuda").bfloat16().float().requires_grad_()
    b = torch.randn(40, generator=gen, device="cuda").bfloat16().float().requires_grad_() if bias else None
    outs = adaln.LinearFunction.apply(x, tx, w, b)
    ref_in = [None if z is None else z.detach().double().requires_grad_() for z in (x, tx, w, b)]
    refs = F.linear(ref_in[0], ref_in[2], ref_in[3]), F.linear(ref_in[1], ref_in[2])
    keep = [i for i, name in enumerate(("y", "ty")) if cot in ("both", name)]
    g = torch.randn(2, 3, 5, 40, generator=gen, device="cuda").bfloat16()
    wrt = [i for i, z in enumerate((x, tx, w, b)) if z is not None]
    got = torch.autograd.grad([outs[i] for i in keep], [(x, tx, w, b)[i] for i in wrt], [g[i] for i in keep],
                              allow_unused=True)
    ref = torch.autograd.grad([refs[i] for i in keep], [ref_in[i] for i in wrt], [g[i].double() for i in keep],
                              allow_unused=True)
    for i in range(2):
        _check(f"output {i}", outs[i], refs[i])
    for i, a, r in zip(wrt, got, ref):
        assert (a is None) == (r is None)
        if a is not None:
            assert a.dtype == (x, tx, w, b)[i].dtype and a.shape == r.shape
            _check(f"gradient {i}", a, r)


@pytest.mark.parametrize("hook", [False, True])
def test_training_step_with_and_without(monkeypatch, hook):
    """Both losses and every gradient through the kernels and through the PyTorch operations; a module with a hook keeps
    its PyTorch operations."""
    torch.manual_seed(0)
    B, S, V = 4, 16, 48
    net = DIT(V, 128, 16, 2, 2, 0.0, S).cuda()
    for p in net.parameters():
        if not p.any():
            torch.nn.init.normal_(p, std=0.05)
    x0, x1 = torch.randn(B, S, V, device="cuda"), torch.randint(0, V, (B, S), device="cuda")
    t = torch.rand(B, device="cuda")
    s = t * torch.rand(B, device="cuda")
    seen = []
    if hook:
        net.blocks[0].norm1.register_forward_hook(lambda *_: seen.append(1))
    calls = []
    for name in ("gated_norm", "chunk", "attention", "gelu"):
        def served(*a, f=getattr(adaln, name)):
            out = f(*a)
            calls.append((f.__name__, out is not None))
            return out
        monkeypatch.setattr(adaln, name, served)

    def step():
        net.zero_grad(set_to_none=True)
        with torch.autocast("cuda", dtype=torch.bfloat16):
            sd = train_step.lag_self_distillation_loss(net, x0[:2], x1[:2], t=t[:2], s=s[:2])
            vf = train_step.vfm_loss(net, x0[2:], x1[2:], t=t[2:])
        (vf + sd).backward()
        return vf.item(), sd.item(), torch.cat([p.grad.flatten() for p in net.parameters()])

    got = step()
    # three network calls; six functions per block and two in the output layer
    assert len(calls) == 3 * (8 if hook else 14) and all(served for _, served in calls), calls
    assert len(seen) == (3 if hook else 0)
    layers = []
    linear = adaln.linear
    monkeypatch.setattr(adaln, "linear", lambda *a: layers.append(linear(*a) is not None) or linear(*a))
    step()
    assert sum(layers) == (7 if hook else 12)  # of the three network calls the one under forward-mode AD
    monkeypatch.setattr(adaln, "serves_block", lambda x: False)
    ref = step()
    # two blocks of bf16 products on either side, each rounding its operands: 2^-9 per product
    assert abs(got[0] - ref[0]) < 1e-2 * abs(ref[0]) and abs(got[1] - ref[1]) < 1e-2 * abs(ref[1])
    assert (got[2] - ref[2]).norm() < 3e-2 * ref[2].norm()


@pytest.mark.parametrize("train", ["net", "dropout only"])
def test_training_step_with_dropout(monkeypatch, train):
    """A training block's dropout goes in front of the gate: the same masks as behind it, the same gradients, also
    where only the dropout modules are in training mode."""
    torch.manual_seed(0)
    B, S, V = 4, 16, 48
    net = DIT(V, 128, 16, 2, 2, 0.3, S).cuda()
    for p in net.parameters():
        if not p.any():
            torch.nn.init.normal_(p, std=0.05)
    if train != "net":
        net.eval()
        for block in net.blocks:
            block.dropout.train()
    x0, x1 = torch.randn(B, S, V, device="cuda"), torch.randint(0, V, (B, S), device="cuda")
    t = torch.rand(B, device="cuda")
    s = t * torch.rand(B, device="cuda")

    def step():
        torch.manual_seed(1)
        net.zero_grad(set_to_none=True)
        with torch.autocast("cuda", dtype=torch.bfloat16):
            vf = train_step.vfm_loss(net, x0[2:], x1[2:], t=t[2:])
            sd = train_step.lag_self_distillation_loss(net, x0[:2], x1[:2], t=t[:2], s=s[:2])
        (vf + sd).backward()
        return vf.item(), sd.item(), torch.cat([p.grad.flatten() for p in net.parameters()])

    calls = []
    norm = adaln.gated_norm
    monkeypatch.setattr(adaln, "gated_norm", lambda *a: (calls.append(1), norm(*a))[1])
    got = step()
    assert len(calls) == 3 * 7
    monkeypatch.setattr(adaln, "serves_block", lambda x: False)
    ref = step()
    # as without dropout; another mask would differ by far more
    assert abs(got[0] - ref[0]) < 1e-2 * abs(ref[0]) and abs(got[1] - ref[1]) < 1e-2 * abs(ref[1])
    assert (got[2] - ref[2]).norm() < 3e-2 * ref[2].norm()
