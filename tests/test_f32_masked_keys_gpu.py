"""Keys of the type's lowest value, whose scores overflow to -inf, take no part wherever they stand among the tiles of the fp32
kernels: whole tiles of them, at the start, at the end (all that one wave of a split group sees) and for some queries only."""
import pytest
import torch

from oracle import attn_jvp_oracle as orc

pytestmark = pytest.mark.gpu
LOWEST = torch.finfo(torch.float32).min
TOL = 1e-5  # the bound that the fp32 mode is held to elsewhere


@pytest.mark.parametrize("some", [False, True])
@pytest.mark.parametrize("B,H,Lq,Lk,D,masked", [
    (1, 2, 40, 40, 64, [(24, 40)]), (1, 2, 40, 64, 64, [(48, 64)]), (1, 2, 33, 200, 36, [(0, 40), (100, 200)]),
    (1, 2, 20, 64, 30, [(0, 16), (32, 63)]), (1, 1, 17, 16, 32, [(0, 12)]), (2, 2, 70, 129, 128, [(0, 112)]),
    (66, 12, 64, 48, 64, [(0, 16), (32, 48)])])  # the last: a wave per group, every key in it
# (several keys stay in each case: with one the gradients of the scores are zero, and what is left is rounding)
def test_lowest_keys(B, H, Lq, Lk, D, masked, some):
    from semicat_amd import kernels as K
    x = orc.make_inputs(B, H, Lq, Lk, D, seed=3, tangent_scale=0.5, dtype=torch.float32)
    # column 0 decides: positive in the queries that see the masked keys at -inf, 0 in the others
    x["q"][..., 0] = 0.0 if some else 8.0
    if some:
        x["q"][:, :, ::3, 0] = 8.0
    for n in ("tq", "tk"):
        x[n][..., 0] = 0.0  # keeps the scores' tangents finite
    x["k"][..., 0] = 0.0
    for a, b in masked:
        x["k"][:, :, a:b, 0] = LOWEST
    c = {n: t.double() for n, t in x.items()}

    def attention(q, k, v):
        return torch.softmax(q @ k.transpose(-1, -2) / D ** 0.5, -1) @ v

    leaves = [c[n].requires_grad_() for n in ("q", "k", "v", "tq", "tk", "tv")]
    o, to = torch.func.jvp(attention, tuple(leaves[:3]), tuple(leaves[3:]))
    grads = torch.autograd.grad((o, to), leaves, (c["dO"], c["dTO"]))
    d = {n: t.cuda() for n, t in x.items()}
    print(f"[masked keys] {(B, H, Lq, Lk, D)} {masked} some={some}", flush=True)
    go, gto, lse, mu, _ = K.attention_jvp_forward(*[d[n] for n in ("q", "k", "v", "tq", "tk", "tv")])
    got = K.attention_jvp_backward(*[d[n] for n in ("q", "k", "v", "tq", "tk", "tv")], go, gto, lse, mu, dO=d["dO"],
                                   dTO=d["dTO"])
    po, _ = K.attention_forward(d["q"], d["k"], d["v"])
    for name, a, r in zip(("o", "to", "primal o", "dq", "dk", "dv", "dtq", "dtk", "dtv"), (go, gto, po, *got),
                          (o, to, o, *grads)):
        a, r = a.cpu().double(), r.detach()
        if name in ("dq", "dtq"):  # column 0 sums products with the lowest value, rounding included
            a, r = a[..., 1:], r[..., 1:]
        assert orc.rel_frobenius(a, r) <= TOL, name  # (also false for NaN)
