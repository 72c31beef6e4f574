"""Modules of a DiT block whose call is not just the forward of their class are called, not passed by. (CPU: the choice of
the path alone.)"""
import pytest
import torch

from semicat_amd import adaln
from semicat_amd.dit import DDiTBlock

NAMES = ("norm1", "norm2", "dropout", "mlp", "mlp.1", "attn_qkv", "attn_out", "mlp.0", "mlp.2", "adaLN_modulation")


def _own_forward(m):
    m.forward = lambda *a, f=m.forward: f(*a)


def _compiled(m):
    m.compile(backend="eager")


@pytest.mark.parametrize("change", [_own_forward, _compiled])
@pytest.mark.parametrize("name", NAMES)
def test_changed_module_is_called(monkeypatch, change, name):
    monkeypatch.setattr(adaln, "serves_block", lambda x: True)
    block = DDiTBlock(16, 2, 4, 8)
    x = torch.randn(2, 4, 16)
    assert block._fuses(x)
    module = block.get_submodule(name)
    x16 = torch.randn(2, module.in_features).bfloat16() if isinstance(module, torch.nn.Linear) else None

    def served():
        if x16 is None:
            return block._fuses(x)
        seen = []
        torch.func.jvp(lambda z: (seen.append(adaln.linear(module, z)), z)[1], (x16,), (x16,))
        return seen[0] is not None

    assert served()
    change(module)
    assert not served()
