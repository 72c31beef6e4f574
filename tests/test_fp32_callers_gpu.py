"""float32 callers of safe_sdpa_jvp: exactly what casting to bfloat16 around the op gives, for every input that such casts
accept, with tensors that the caller may write to afterwards and no more memory kept for the backward."""
import pytest
import torch

from semicat_amd import safe_sdpa_jvp

pytestmark = pytest.mark.gpu


def _casts(q, k, v):
    return safe_sdpa_jvp(q.bfloat16(), k.bfloat16(), v.bfloat16()).to(q.dtype)


def _inputs(B, S, H, D, dtype=torch.float32):
    gen = torch.Generator("cuda").manual_seed(S + D)
    x = [(torch.randn(B, S, H, D, device="cuda", generator=gen) * s).to(dtype).requires_grad_()
         for s in (1.0, 1.0, 1.0, 0.1, 0.1, 0.1)]
    return x, [torch.randn(B, S, H, D, device="cuda", generator=gen).to(dtype) for _ in range(2)]


def _step(fn, x, g, jvp):
    if not jvp:
        y = fn(*x[:3])
        return y, *torch.autograd.grad(y, x[:3], g[0])
    y, ty = torch.func.jvp(fn, tuple(x[:3]), tuple(x[3:]))
    return y, ty, *torch.autograd.grad((y, ty), x, g)


@pytest.mark.parametrize("jvp", [False, True])
@pytest.mark.parametrize("B,S,H,D,dtype", [
    (2, 128, 4, 64, torch.float32), (2, 77, 3, 32, torch.float32), (1, 300, 2, 128, torch.float32),
    (2, 200, 2, 36, torch.float32), (2, 40, 2, 64, torch.float64)])
def test_same_bits_as_casts(B, S, H, D, dtype, jvp):
    x, g = _inputs(B, S, H, D, dtype)
    for a, b in zip(_step(safe_sdpa_jvp, x, g, jvp), _step(_casts, x, g, jvp)):
        assert a.dtype == dtype and a.stride() == b.stride() and torch.equal(a, b)


@pytest.mark.parametrize("jvp", [False, True])
@pytest.mark.parametrize("layout", [
    lambda t: t.repeat_interleave(2, dim=-1)[..., ::2],       # every second column of a wider tensor
    lambda t: t[..., :1].expand(t.shape),                     # one column read by all
    lambda t: t[:, :, :1].expand(t.shape)])                   # one head read by all
def test_layouts_without_unit_stride(layout, jvp):
    x, g = _inputs(2, 48, 3, 64)
    x = [layout(t.detach()).requires_grad_() for t in x]
    for a, b in zip(_step(safe_sdpa_jvp, x, g, jvp), _step(_casts, x, g, jvp)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("jvp", [False, True])
def test_inputs_and_result_may_be_written_to(jvp):
    x, g = _inputs(2, 48, 3, 64)
    ref = _step(_casts, x, g, jvp)
    kept = []

    def fn(*qkv):
        own = [t * 1.0 for t in qkv]
        y = safe_sdpa_jvp(*own)
        out = y + 0.0
        for t in (y, *own):
            kept.append(t.mul_(3.0))
        return out

    for a, b in zip(_step(fn, x, g, jvp), ref):
        assert torch.equal(a, b)
    assert len(kept) == 4


@pytest.mark.parametrize("jvp", [False, True])
def test_memory_kept_for_the_backward(jvp):
    x, g = _inputs(8, 256, 8, 64)
    held = []
    for fn in (_casts, safe_sdpa_jvp):
        torch.cuda.synchronize()
        before = torch.cuda.memory_allocated()
        if jvp:
            out = torch.func.jvp(lambda *a: fn(*[t * 1.0 for t in a]), tuple(x[:3]), tuple(x[3:]))
        else:
            out = fn(*[t * 1.0 for t in x[:3]])
        held.append(torch.cuda.memory_allocated() - before)
        del out
    assert held[1] <= held[0]
