"""Head dimensions that end ahead of their class's last tiles: the kernels leave the tiles beyond them out.  The sizes on both
sides of each line, aligned and unaligned rows, launches of few and of many workgroups, one and several sets of rows a wave."""
import pytest
import torch

from oracle import attn_jvp_oracle as orc

pytestmark = pytest.mark.gpu
ORDER = ("q", "k", "v", "tq", "tk", "tv")
GRADS = ("dq", "dk", "dv", "dtq", "dtk", "dtv")


# the bound of the other parity tests, by the unit roundoff of the type (2^-8 and 2^-11)
BOUND = {torch.bfloat16: 1e-2, torch.float16: 1e-2 / 8}
SIZES = (16, 17, 24, 33, 40, 47, 48, 49, 56, 65, 72, 80, 95, 96, 97, 104)
# (wide waves take 16-byte aligned rows, and two sizes on a side are enough)
CASES = [(*shape, D) for shape in ((1, 2, 90, 70), (1, 3, 300, 170), (8, 12, 77, 333)) for D in SIZES] + \
        [(*shape, D) for shape in ((1, 150, 200, 260), (2, 300, 130, 257)) for D in (16, 40, 48, 80, 96)]


@pytest.mark.parametrize("B,H,Lq,Lk,D", CASES)
@pytest.mark.parametrize("mode", ["both", "dO", "dTO", "primal"])
def test_head_dimensions_at_the_edges_of_tiles(B, H, Lq, Lk, D, mode):
    from semicat_amd import kernels as K
    print(f"[tiles] {B} {H} {Lq} {Lk} {D} {mode}", flush=True)
    dtype = torch.float16 if (D + Lq) % 2 else torch.bfloat16
    x = orc.make_inputs(B, H, Lq, Lk, D, seed=Lq + D, tangent_scale=0.3, dtype=dtype)
    d = {n: t.cuda() for n, t in x.items()}
    a = [d[n] for n in ORDER]
    dO, dTO = mode != "dTO", mode in ("both", "dTO")
    if mode == "primal":
        o, lse = K.attention_forward(*a[:3])
        to = mu = None
        g = K.attention_jvp_backward(*a[:3], None, None, None, o, None, lse, None, dO=d["dO"])
    else:
        o, to, lse, mu, _ = K.attention_jvp_forward(*a)
        g = K.attention_jvp_backward(*a, o, to, lse, mu, dO=d["dO"] if dO else None, dTO=d["dTO"] if dTO else None)
    few = min(B * H, 6)  # heads that the oracle forms: the first and the last
    heads = torch.cat((torch.arange(few // 2), torch.arange(B * H - (few - few // 2), B * H)))
    pick = {n: t.reshape(1, B * H, *t.shape[2:])[:, heads] for n, t in x.items()}
    ref = orc.attention_jvp_autograd(*[pick[n] for n in ORDER], dO=pick["dO"] if dO else None, dTO=pick["dTO"] if dTO else None)
    for n, t in {"O": o, "TO": to, **dict(zip(GRADS, g))}.items():
        if t is None or n not in ref:
            continue
        got = t.cpu().reshape(1, B * H, *t.shape[2:])
        assert torch.isfinite(got.float()).all(), n
        err = orc.rel_frobenius(got[:, heads], ref[n])
        assert err <= BOUND[dtype], (n, err)
