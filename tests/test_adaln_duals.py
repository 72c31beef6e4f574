"""Outputs of the DiT's fused functions become dual tensors without a copy: the tangent keeps the memory it was written
to.  (CPU; the launches are stubs, the memory they would fill is what is looked at.)"""
import pytest
import torch
from torch import nn

from semicat_amd import adaln, functional, kernels

B, S, W, H = 2, 5, 16, 2


def _modulation(x):
    """The modulation as the block makes it: chunks of a linear layer's output."""
    return adaln.chunk(adaln.linear(nn.Linear(W, 6 * W), x[:, 0]), 6)


def _gated_norm(x):
    gate, scale, shift, *_ = _modulation(x)
    return adaln.gated_norm(x, x, gate, nn.LayerNorm(W), scale, shift)


CALLS = {
    "linear": lambda x: adaln.linear(nn.Linear(W, 24), x),
    "linear without bias": lambda x: adaln.linear(nn.Linear(W, 24, bias=False), x),
    "two linear layers": lambda x: adaln.linear(nn.Linear(24, 8, bias=False), adaln.linear(nn.Linear(W, 24), x)),
    "chunks": _modulation,
    "gelu": lambda x: adaln.gelu(adaln.linear(nn.Linear(W, 24), x)),
    "gated norm": _gated_norm,
    "attention": lambda x: adaln.attention(
        adaln.linear(nn.Linear(W, 3 * 2 * W, bias=False), x).view(B, S, 3, H, W), torch.ones(S, W // 2),
        torch.zeros(S, W // 2)),
}


@pytest.mark.parametrize("name", CALLS)
def test_no_copy_behind_make_dual(monkeypatch, name):
    monkeypatch.setattr(adaln, "_launch", lambda *a: None)
    monkeypatch.setattr(adaln, "_gelu", lambda *a: None)
    monkeypatch.setattr(torch.Tensor, "is_cuda", True, raising=False)
    monkeypatch.setattr(kernels, "rotary_fusable", lambda *a, **k: True)
    monkeypatch.setattr(kernels, "attention_jvp_forward", lambda *a, **k: (None, None, torch.zeros(1), torch.zeros(1), None))
    seen = []

    def dual(interpreter, primal, tangent, make=functional._dual_above):
        before = tangent.data_ptr()
        out = make(interpreter, primal, tangent)
        kept = functional._below_jvp([out])[1][0][1]
        seen.append(kept.data_ptr() == before and kept.grad_fn is not None
                    and "Copy" not in kept.grad_fn.name())
        return out

    monkeypatch.setattr(adaln, "_dual_above", dual)
    torch.manual_seed(0)
    x = torch.randn(B, S, W).bfloat16()
    with torch.autocast("cpu", dtype=torch.bfloat16):
        torch.func.jvp(CALLS[name], (x,), (torch.ones_like(x).requires_grad_(),))
    assert seen and all(seen), seen
