"""What the gated residual and norm keep for the backward: nothing that their reverse mode does not read, so that a block's
output may be written to.  (CPU; the launches are stubs.)"""
import pytest
import torch

from semicat_amd import adaln

B, S, W = 2, 3, 16


@pytest.mark.parametrize("mode", ["gate", "norm", "both"])
@pytest.mark.parametrize("jvp", [False, True])
def test_saved_tensors(monkeypatch, mode, jvp):
    calls = []
    monkeypatch.setattr(adaln, "_launch", lambda fn, j, shape, eps, t: calls.append((fn, tuple(shape), t)))
    gate, norm = mode != "norm", mode != "gate"
    act = lambda on: torch.randn(B, S, W).bfloat16().requires_grad_() if on else None
    mod = lambda on: torch.randn(B, 1, W).bfloat16().requires_grad_() if on else None
    vec = lambda on: torch.randn(W).requires_grad_() if on else None
    t = [act(True), act(gate), mod(gate), mod(norm), mod(norm), vec(norm), vec(norm), act(jvp), act(gate and jvp),
         mod(gate and jvp), mod(norm and jvp), mod(norm and jvp)]
    kept = []
    with torch.autograd.graph.saved_tensors_hooks(lambda z: kept.append(z) or z, lambda z: z):
        y, h, ty, th = adaln.GatedNormFunction.apply(1e-5, jvp, *t)
    whole = sum(z.shape == (B, S, W) for z in kept)
    # norm alone: its input; with a gate the gated tensor and, in front of a norm, y; each with its tangent
    assert whole == (2 if mode == "both" else 1) * (2 if jvp else 1)
    outs = [z for z in ((y, ty) if mode == "gate" else (h, th)) if z is not None]
    with torch.no_grad():
        for z in outs + ([t[0]] if gate else []):
            z.mul_(2.0)
    wrt = [z for z in t if z is not None]
    grads = torch.autograd.grad(outs, wrt, [torch.ones_like(z) for z in outs], allow_unused=True)
    fn, shape, given = calls[-1]
    assert fn == "sjvp_adaln_bwd" and shape == (B, S, W) and given["x"] is not None
    assert (given["y"] is not None) == (mode == "both")
    for z, g in zip(wrt, grads):
        assert g.shape == z.shape and g.dtype == z.dtype
