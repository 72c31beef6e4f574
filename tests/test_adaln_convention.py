"""The reverse mode of the tangent of a modulated LayerNorm holds the mean and the reciprocal deviation of its input constant.
Written out in fp64 here, so that the kernels are held to the formula and not to what PyTorch's layer_norm does."""
import pytest
import torch
import torch.nn.functional as F


def _written_out(y, ty, w, b, scale, tscale, shift, tshift, eps, constant=True):
    """h and its tangent; ``constant``: the statistics are constants of the tangent."""
    mean = y.mean(-1, keepdim=True)
    r = (y.var(-1, unbiased=False, keepdim=True) + eps).rsqrt()
    h = (y - mean) * r * w + b
    if constant:
        mean, r = mean.detach(), r.detach()
    centred = ty - ty.mean(-1, keepdim=True)
    xhat = (y - mean) * r
    # the primal's normalised rows where the tangent only scales them, with their own derivative
    th = r * (centred - xhat * (centred * xhat).mean(-1, keepdim=True)) * w
    return h * (1 + scale) + shift, th * (1 + scale) + h * tscale + tshift


def _inputs(B, S, W, device, dtype):
    gen = torch.Generator(device).manual_seed(W)
    act = [torch.randn(B, S, W, device=device, generator=gen).to(dtype).requires_grad_() for _ in range(2)]
    vec = [torch.randn(W, device=device, generator=gen, dtype=torch.float64 if dtype == torch.float64 else None).requires_grad_()
           for _ in range(2)]
    mod = [(torch.randn(B, 1, W, device=device, generator=gen) * 0.5).to(dtype).requires_grad_() for _ in range(4)]
    cot = [torch.randn(B, S, W, device=device, generator=gen).to(dtype) for _ in range(2)]
    return act, vec, mod, cot


def test_pytorch_has_the_same_convention_here():
    (y, ty), (w, b), (scale, tscale, shift, tshift), cot = _inputs(2, 3, 16, "cpu", torch.float64)
    outs = torch.func.jvp(lambda y, scale, shift: F.layer_norm(y, (16,), w, b, 1e-5) * (1 + scale) + shift,
                          (y, scale, shift), (ty, tscale, tshift))
    wrt = (y, ty, w, b, scale, tscale, shift, tshift)
    got = torch.autograd.grad(outs, wrt, cot)
    same, other = (torch.autograd.grad(_written_out(y, ty, w, b, scale, tscale, shift, tshift, 1e-5, constant), wrt, cot)
                   for constant in (True, False))
    for g, r in zip(got, same):
        torch.testing.assert_close(g, r, rtol=1e-9, atol=1e-9)
    assert (other[0] - same[0]).norm() > 1e-2 * same[0].norm()  # the full derivative is another


@pytest.mark.gpu
@pytest.mark.parametrize("B,S,W", [(2, 5, 24), (3, 17, 768)])
def test_kernels_have_the_written_out_convention(B, S, W):
    from semicat_amd import adaln
    (y, ty), (w, b), (scale, tscale, shift, tshift), cot = _inputs(B, S, W, "cuda", torch.bfloat16)
    _, h, _, th = adaln.GatedNormFunction.apply(1e-5, True, y, None, None, scale, shift, w, b, ty, None, None, tscale, tshift)
    wrt = (y, ty, w, b, scale, tscale, shift, tshift)
    got = (h, th, *torch.autograd.grad((h, th), wrt, cot))
    d = [z.detach().double().requires_grad_() for z in wrt]
    outs = _written_out(*d, 1e-5)
    ref = (*outs, *torch.autograd.grad(outs, d, [c.double() for c in cot]))
    for i, (g, r) in enumerate(zip(got, ref)):
        # every result is rounded to bf16 once: 2^-9 at most, 2^-9 / sqrt(3) in the root mean square
        assert (g.double() - r).norm() < 4e-3 * r.norm(), i
