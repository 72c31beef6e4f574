"""The op computed below torch.func.jvp's level against the same call through functorch's general dispatch."""
import pytest
import torch

from semicat_amd import functional
from tests import eager_backend


def _run(x, g, wrapped, cot, grad_mode=True, hooks=None, op=None):
    """Outputs and gradients; ``wrapped`` says which of q, k, v carry a tangent (the others are constants)."""
    x = [t.detach().clone().requires_grad_() for t in x]

    def f(*dual):
        dual = iter(dual)
        return (op or functional.safe_sdpa_jvp)(*[next(dual) if w else t for w, t in zip(wrapped, x[:3])])

    primals = tuple(t for w, t in zip(wrapped, x[:3]) if w)
    tangents = tuple(t for w, t in zip(wrapped, x[3:]) if w)
    with torch.set_grad_enabled(grad_mode):
        if hooks:
            with torch.autograd.graph.saved_tensors_hooks(*hooks):
                y, ty = torch.func.jvp(f, primals, tangents)
        else:
            y, ty = torch.func.jvp(f, primals, tangents)
    if not grad_mode:
        return y, ty
    outs, cots = zip(*[(o, c) for o, c, name in ((y, g[0], "y"), (ty, g[1], "ty")) if cot in ("both", name)])
    return y, ty, *torch.autograd.grad(outs, x, cots, allow_unused=True)


def _inputs(dtype=torch.float32):
    gen = torch.Generator().manual_seed(5)
    x = [torch.randn(2, 9, 3, 16, generator=gen, dtype=dtype) for _ in range(6)]
    return x, [torch.randn(2, 9, 3, 16, generator=gen, dtype=dtype) for _ in range(2)]


def _both(monkeypatch, run):
    a = run()
    with monkeypatch.context() as m:
        m.setattr(functional, "_below_jvp", lambda tensors: None)
        b = run()
    assert len(a) == len(b)
    for s, t in zip(a, b):
        assert (s is None) == (t is None)
        if s is not None:
            assert s.dtype == t.dtype and s.shape == t.shape and s.stride() == t.stride()
            torch.testing.assert_close(s, t, rtol=0, atol=0)
    return a


@pytest.mark.parametrize("wrapped", [(1, 1, 1), (1, 0, 1), (0, 1, 0)])
@pytest.mark.parametrize("cot", ["both", "y", "ty"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_same_values_and_gradients(monkeypatch, wrapped, cot, dtype):
    eager_backend.install(monkeypatch)
    x, g = _inputs(dtype)
    _both(monkeypatch, lambda: _run(x, g, wrapped, cot))


def test_route_taken_only_under_one_jvp(monkeypatch):
    eager_backend.install(monkeypatch)
    x, g = _inputs()
    seen = []
    real = functional._below_jvp

    def spy(tensors):
        seen.append(real(tensors))
        return seen[-1]

    monkeypatch.setattr(functional, "_below_jvp", spy)
    functional.safe_sdpa_jvp(*x[:3])
    assert seen.pop() is None
    torch.func.jvp(functional.safe_sdpa_jvp, tuple(x[:3]), tuple(x[3:]))
    assert seen.pop() is not None

    def inner(*p):
        return torch.func.jvp(functional.safe_sdpa_jvp, p, tuple(x[3:]))[1]

    try:
        torch.func.vjp(inner, *x[:3])
    except Exception:  # whatever the general dispatch makes of a second transform
        pass
    assert all(s is None for s in seen)


def test_saved_tensor_hooks_and_no_grad(monkeypatch):
    eager_backend.install(monkeypatch)
    x, g = _inputs()
    packed = []

    def pack(t):
        packed.append(t.shape)
        return t.clone()

    _both(monkeypatch, lambda: _run(x, g, (1, 1, 1), "both", hooks=(pack, lambda t: t)))
    assert packed
    y, ty = _both(monkeypatch, lambda: _run(x, g, (1, 1, 1), "both", grad_mode=False))
    assert not y.requires_grad and not ty.requires_grad


@pytest.mark.parametrize("wrapped", [(1, 1, 1), (1, 0, 1), (0, 1, 0), (0, 0, 1)])
@pytest.mark.parametrize("cot", ["both", "y", "ty"])
@pytest.mark.parametrize("dtype,rot", [(torch.bfloat16, 16), (torch.float16, 8), (torch.float32, 16)])
def test_rotation_in_front_of_the_kernels(monkeypatch, wrapped, cot, dtype, rot):
    """Shapes that the folded rotation does not serve, a part of the head dimension rotated among them."""
    eager_backend.install(monkeypatch)
    x, g = _inputs(dtype)
    cos, sin = torch.randn(2, 11, rot // 2, generator=torch.Generator().manual_seed(1))
    _both(monkeypatch, lambda: _run(x, g, wrapped, cot, op=lambda q, k, v: functional.safe_sdpa_jvp_rotary(q, k, v, cos, sin)))
