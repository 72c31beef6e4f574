"""tanh GELU and its derivatives over every bf16 value that PyTorch's own kernels serve with finite results."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tangent", [1.0, 0.0, -3.0])
def test_every_bf16_value(tangent):
    from semicat_amd import adaln
    u = torch.arange(65536, device="cuda", dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    u = u[u.float().abs() <= 1.8e13]
    u = u[:u.numel() // 8 * 8].clone().requires_grad_()
    tu = torch.full_like(u, tangent).requires_grad_()
    cot = torch.full_like(u, 1.0), torch.full_like(u, 0.5)
    outs = adaln.GeluFunction.apply(u, tu)
    got = (*outs, *torch.autograd.grad(outs, (u, tu), cot))
    u64, tu64 = (z.detach().double().requires_grad_() for z in (u, tu))
    refs = torch.func.jvp(lambda z: F.gelu(z, approximate="tanh"), (u64,), (tu64,))
    ref = (*refs, *torch.autograd.grad(refs, (u64, tu64), [c.double() for c in cot]))
    for name, g, r in zip(("y", "ty", "du", "dtu"), got, ref):
        assert g.isfinite().all(), name
        # one rounding to bf16, 2^-9 of the value; 1 + tanh cancels for negative values, to 1e-6 of u and of the tangent
        assert ((g.double() - r).abs() <= 2.0 ** -8 * r.abs() + 4e-6 * (u64.abs() + abs(tangent) + 1)).all(), name
