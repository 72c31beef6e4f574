"""The kernels whose wavefronts own 32 positions, which many workgroups of them have to ask for: forward and row-owned
backward without tangents, column-owned backward without tangents and at head dimensions up to 32."""
import pytest
import torch

from oracle import attn_jvp_oracle as orc

pytestmark = pytest.mark.gpu
ORDER = ("q", "k", "v", "tq", "tk", "tv")


# the bound of the other parity tests, by the unit roundoff of the type (2^-8 and 2^-11)
BOUND = {torch.bfloat16: 1e-2, torch.float16: 1e-2 / 8}
# (batch * heads, Lq, Lk): a wave whose second 16 rows do not exist, workgroups with waves without rows, key axes that end
# inside a tile, a stage, a wave's rows
SHAPES = ((512, 257, 259), (512, 272, 305), (342, 300, 383), (128, 513, 1029))
SIZES = ((64, torch.bfloat16), (48, torch.float16), (32, torch.bfloat16), (24, torch.float16), (128, torch.bfloat16), (72, torch.float16))
CASES = [(*shape, *size, "primal") for shape in SHAPES for size in SIZES] + \
        [(*SHAPES[3], *size, mode) for size in SIZES[2:4] for mode in ("dO", "both")]  # with tangents: the column kernel, D <= 32


@pytest.mark.parametrize("BH,Lq,Lk,D,dtype,mode", CASES)
def test_waves_of_32_rows(BH, Lq, Lk, D, dtype, mode):
    from semicat_amd import kernels as K
    print(f"[wide] {BH} {Lq} {Lk} {D} {dtype} {mode}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(Lq + D)
    x = {n: (torch.randn((1, BH, Lk if n in ("k", "v", "tk", "tv") else Lq, D), device="cuda", generator=gen)
             * (0.3 if n.startswith("t") else 1.0)).to(dtype) for n in (*ORDER, "dO", "dTO")}
    if mode == "primal":
        o, lse = K.attention_forward(*[x[n] for n in ORDER[:3]])
        grads = K.attention_jvp_backward(*[x[n] for n in ORDER[:3]], None, None, None, o, None, lse, None, dO=x["dO"])
        res = {"O": o, **dict(zip(("dq", "dk", "dv"), grads))}
    else:
        o, to, lse, mu, _ = K.attention_jvp_forward(*[x[n] for n in ORDER])
        grads = K.attention_jvp_backward(*[x[n] for n in ORDER], o, to, lse, mu, dO=x["dO"],
                                         dTO=x["dTO"] if mode == "both" else None)
        res = {n: t for n, t in zip(("O", "TO", "dq", "dk", "dv", "dtq", "dtk", "dtv"), (o, to, *grads)) if t is not None}
    # on single heads, against fp64
    for h in (0, 1, BH // 2, BH - 1):
        one = {n: t[:, h:h + 1].cpu() for n, t in x.items()}
        ref = orc.attention_jvp_autograd(*[one[n] for n in ORDER], dO=one["dO"], dTO=one["dTO"] if mode == "both" else None)
        for n, t in res.items():
            err = orc.rel_frobenius(t[:, h:h + 1].cpu(), ref[n])
            assert err <= BOUND[dtype], (h, n, err)  # (also false for NaN)
        assert torch.allclose(lse[0, h, :Lq].cpu().double(), torch.logsumexp(
            one["q"][0, 0].double() @ one["k"][0, 0].double().T * D ** -0.5, -1), rtol=2e-5, atol=2e-5)
