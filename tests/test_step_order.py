"""Both losses of a step in one autocast context, in either order: the gradients are the same."""
import torch

from semicat_amd import train_step as ts
from semicat_amd.dit import DIT, math_attention


def test_order_of_the_two_losses_under_autocast():
    torch.manual_seed(0)
    net = DIT(vocab_size=20, hidden_size=32, cond_dim=16, n_blocks=2, n_heads=2, dropout=0.0, length=8,
              attention_override=math_attention, rotary="torch")
    for p in net.parameters():
        torch.nn.init.normal_(p, std=0.1)
    x0, x1 = torch.randn(4, 8, 20), torch.randint(0, 20, (4, 8))
    t = torch.rand(4)
    s = t * torch.rand(4)

    def grads(order):
        net.zero_grad(set_to_none=True)
        with torch.autocast("cpu", dtype=torch.bfloat16):
            losses = [ts.vfm_loss(net, x0, x1, t=t) if o == "vfm" else
                      ts.lag_self_distillation_loss(net, x0, x1, t=t, s=s) for o in order]
        sum(losses).backward()
        return {n: p.grad.clone() for n, p in net.named_parameters()}

    a, b = grads(("vfm", "sd")), grads(("sd", "vfm"))
    for n in a:
        assert (a[n] - b[n]).norm() <= 2e-2 * a[n].norm(), n  # bf16: sums in another order


def test_losses_on_a_device_without_autocast():
    """Shapes and operation counts are taken on the meta device, which has no autocast at all."""
    with torch.device("meta"):
        net = DIT(vocab_size=20, hidden_size=32, cond_dim=16, n_blocks=1, n_heads=2, dropout=0.0, length=8,
                  attention_override=math_attention, rotary="torch")
        x0, x1, t = torch.randn(4, 8, 20), torch.zeros(4, 8, dtype=torch.long), torch.rand(4)
        loss = ts.lag_self_distillation_loss(net, x0, x1, t=t, s=t * torch.rand(4)) + ts.vfm_loss(net, x0, x1, t=t)
    loss.backward()
    assert all(p.grad is not None and p.grad.shape == p.shape for p in net.parameters())
