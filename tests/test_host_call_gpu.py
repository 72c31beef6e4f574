"""The host extension serves a call exactly as the general form of the entry points does: same results, same
layouts, and whatever it does not serve ends in the general form's own errors."""
import pytest
import torch

from semicat_amd import kernels

pytestmark = pytest.mark.gpu


def _inputs(B, H, Lq, Lk, D, dtype, seq_major=False, offset=0):
    gen = torch.Generator(device="cuda").manual_seed(3)

    def make(L, scale):
        shape = (B, L, H, D) if seq_major else (B, H, L, D)
        n = B * L * H * D
        t = (torch.randn(n + offset, device="cuda", generator=gen) * scale).to(dtype)[offset:].view(shape)
        return t.transpose(1, 2) if seq_major else t

    return [make(L, s) for L, s in ((Lq, 1.0), (Lk, 1.0), (Lk, 1.0), (Lq, 0.1), (Lk, 0.1), (Lk, 0.1), (Lq, 1.0), (Lq, 1.0))]


def _step(x, has_do, has_g, arithmetic=None, rope=None, scale=None, given=False):
    q, k, v, tq, tk, tv, dO, dTO = x
    kw = {"arithmetic": arithmetic, "rope": rope, "scale": scale}
    fw = {"o": torch.zeros_like(q), "to": torch.zeros_like(q)} if given else {}
    o, to, lse, mu, li = kernels.attention_jvp_forward(q, k, v, tq, tk, tv, with_li=given, **fw, **kw)
    bw = {}
    if given:
        bw["grads"] = tuple(torch.zeros_like(t) for t in x[:6])
        if rope is None:
            bw["workspace"] = torch.empty(1 << 20, device="cuda", dtype=torch.uint8)
    grads = kernels.attention_jvp_backward(q, k, v, tq, tk, tv, o, to, lse, mu, dO=dO if has_do else None,
                                           dTO=dTO if has_g else None, **bw, **kw)
    po, plse = kernels.attention_forward(q, k, v, **kw)
    return (o, to, lse, mu, li, *grads, po, plse)


@pytest.mark.parametrize("shape,dtype,seq_major,offset,arithmetic", [
    ((2, 3, 40, 40, 32), torch.float16, False, 0, None),
    ((2, 3, 33, 77, 36), torch.bfloat16, True, 0, None),
    ((1, 2, 129, 65, 20), torch.bfloat16, False, 3, None),
    ((2, 2, 50, 50, 64), torch.float32, True, 0, None),
    ((2, 2, 50, 50, 64), torch.float32, True, 0, "bf16"),
    ((2, 2, 128, 128, 64), torch.bfloat16, True, 0, "bf16"),
])
@pytest.mark.parametrize("cot", ["both", "dO", "dTO"])
@pytest.mark.parametrize("given", [False, True])
def test_host_extension_equals_the_general_form(monkeypatch, shape, dtype, seq_major, offset, arithmetic, cot, given):
    x = _inputs(*shape, dtype, seq_major, offset)
    args = (x, cot != "dTO", cot != "dO", arithmetic, None, 0.2 if given else None, given)
    res = _step(*args)
    monkeypatch.setattr(kernels, "_on_gpu", lambda q: False)
    ref = _step(*args)
    for a, b in zip(res, ref):
        assert (a is None) == (b is None)
        if a is not None:
            assert a.stride() == b.stride() and a.dtype == b.dtype and torch.equal(a, b)


def test_host_extension_with_the_rotation_folded_in(monkeypatch):
    x = _inputs(2, 3, 100, 100, 64, torch.bfloat16, True)
    rope = tuple(torch.randn(128, 32, device="cuda") for _ in range(2))
    res = _step(x, True, True, rope=rope)
    monkeypatch.setattr(kernels, "_on_gpu", lambda q: False)
    for a, b in zip(res, _step(x, True, True, rope=rope)):
        assert (a is None and b is None) or torch.equal(a, b)


def _no_unit_stride(x):
    x[1] = x[1].transpose(2, 3).contiguous().transpose(2, 3)


@pytest.mark.parametrize("spoil,error", [
    (lambda x: x.__setitem__(1, x[1][:, :1]), AssertionError),
    (lambda x: x.__setitem__(4, x[4].half()), TypeError),
    (lambda x: x.__setitem__(2, x[2].cpu()), ValueError),
    (lambda x: x.__setitem__(0, x[0].double()), TypeError),
    (lambda x: x.__setitem__(3, None), AttributeError),
    (_no_unit_stride, AssertionError),
    (lambda x: x.__setitem__(slice(0, 8), [t[..., :8] for t in x]), ValueError),
])
def test_malformed_calls_raise_as_before(spoil, error):
    x = _inputs(2, 3, 32, 32, 32, torch.bfloat16)
    spoil(x)
    with pytest.raises(error):
        kernels.attention_jvp_forward(*x[:6])


def test_refused_scales_and_expanded_inputs(monkeypatch):
    x = _inputs(2, 3, 32, 32, 32, torch.bfloat16)
    for scale in (-1.0, float("inf"), float("nan"), 0.0):
        with pytest.raises(ValueError):
            kernels.attention_jvp_forward(*x[:6], scale=scale)
    x[1] = x[1][:1, :1].expand(2, 3, 32, 32)  # one head read by all: gradients still come per head
    res = _step(x, True, True)
    monkeypatch.setattr(kernels, "_on_gpu", lambda q: False)
    for a, b in zip(res, _step(x, True, True)):
        assert (a is None and b is None) or (torch.equal(a, b) and a.stride() == b.stride())


@pytest.mark.parametrize("n,D,half,dtype,out_dtype,inverse", [
    (4, 64, 32, torch.bfloat16, None, False), (2, 128, 32, torch.bfloat16, torch.float32, True),
    (1, 20, 10, torch.float16, None, True), (3, 48, 0, torch.float32, torch.bfloat16, False)])
def test_rotation_through_the_host_extension(monkeypatch, n, D, half, dtype, out_dtype, inverse):
    fused = torch.randn(2, 33, n, 3, D, device="cuda").to(dtype)
    xs = fused.unbind(2)
    tables = (None, None) if half == 0 else tuple(torch.randn(40, 3 * half, device="cuda")[:, :half] for _ in range(2))
    res = kernels.rotary_embedding(xs, *tables, out_dtype=out_dtype, inverse=inverse)
    monkeypatch.setattr(kernels, "_on_gpu", lambda q: False)
    for a, b in zip(res, kernels.rotary_embedding(xs, *tables, out_dtype=out_dtype, inverse=inverse), strict=True):
        assert torch.equal(a, b) and a.stride() == b.stride() and a.dtype == b.dtype


@pytest.mark.parametrize("how", ["a dispatch mode", "deterministic fill"])
def test_results_that_have_to_be_seen_or_filled_are_made_by_the_dispatcher(how):
    """Their values and strides are those of results that come straight from the allocator."""
    from torch.utils._python_dispatch import TorchDispatchMode
    x = _inputs(2, 3, 33, 77, 64, torch.bfloat16, True)
    x[1] = x[1].transpose(1, 2).contiguous().transpose(1, 2)[:, :1].expand(-1, 3, -1, -1)  # no dense strides to keep
    cos, sin = torch.randn(2, 40, 32, device="cuda")

    def run():
        return (*_step(x, True, True), *kernels.rotary_embedding((x[0].transpose(1, 2),), cos, sin))

    made = []

    class Watch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            made.append(str(func))
            return func(*args, **(kwargs or {}))

    ref = run()
    if how == "a dispatch mode":
        with Watch():
            res = run()
        # o, to, lse, mu, six gradients, workspace, plain o and lse, one rotated tensor
        assert sum("empty" in n for n in made) == 14, made
    else:
        torch.use_deterministic_algorithms(True)
        try:
            assert torch.utils.deterministic.fill_uninitialized_memory
            res = run()
        finally:
            torch.use_deterministic_algorithms(False)
    for a, b in zip(res, ref, strict=True):
        assert (a is None and b is None) or (a.stride() == b.stride() and torch.equal(a, b))
