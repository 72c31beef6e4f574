"""The 16-bit kernels in which several wavefronts share a group of rows, which launches of few workgroups take: every part's
remainder, groups and waves without rows, and keys without a probability in a part."""
import pytest
import torch

from oracle import attn_jvp_oracle as orc

pytestmark = pytest.mark.gpu
ORDER = ("q", "k", "v", "tq", "tk", "tv")
GRADS = ("dq", "dk", "dv", "dtq", "dtk", "dtv")
# the bound of the other parity tests, by the unit roundoff of the type (2^-8 and 2^-11)
BOUND = {torch.bfloat16: 1e-2, torch.float16: 1e-2 / 8}


def _run(x, mode):
    from semicat_amd import kernels as K
    d = {n: t.cuda() for n, t in x.items()}
    a = [d[n] for n in ORDER]
    if mode == "primal":
        o, lse = K.attention_forward(*a[:3])
        g = K.attention_jvp_backward(*a[:3], None, None, None, o, None, lse, None, dO=d["dO"])
        res = {"O": o, **dict(zip(GRADS, g)), "lse": lse}
    else:
        o, to, lse, mu, li = K.attention_jvp_forward(*a)
        g = K.attention_jvp_backward(*a, o, to, lse, mu, dO=None if mode == "dTO" else d["dO"],
                                     dTO=None if mode == "dO" else d["dTO"])
        res = {"O": o, "TO": to, **dict(zip(GRADS, g)), "lse": lse, "mu": mu, "li": li}
    return {n: t.cpu() for n, t in res.items() if t is not None}


# (heads, Lq, Lk): four parts of every kernel with 5 .. 9 stages; two parts of the forward and the pair; two workgroups to a
# compute unit of the pair; one stage more than the parts hold, a stage of one key
@pytest.mark.parametrize("H,Lq,Lk", [(2, 129, 129), (1, 257, 161), (3, 17, 288), (24, 200, 205), (24, 130, 257), (9, 1000, 400),
                                     (30, 500, 513)])
@pytest.mark.parametrize("D,dtype,step", [(64, torch.bfloat16, 1), (32, torch.float16, 1), (48, torch.bfloat16, 1),
                                          (36, torch.bfloat16, 1), (21, torch.float16, 1), (64, torch.float16, 3)])
@pytest.mark.parametrize("mode", ["both", "dO", "dTO", "primal"])
def test_parts_of_a_group(H, Lq, Lk, D, dtype, step, mode):
    print(f"[split] {H} {Lq} {Lk} {D} {dtype} {mode}", flush=True)
    x = orc.make_inputs(1, H, Lq, Lk, D, seed=Lq + D, tangent_scale=0.3, dtype=dtype)
    if step > 1:  # rows that no 16-byte boundary fits
        x = {n: torch.cat((t, t[..., :1]), -1)[..., :-1] for n, t in x.items()}
    ref = orc.attention_jvp_autograd(*[x[n] for n in ORDER], dO=None if mode == "dTO" else x["dO"],
                                     dTO=None if mode in ("dO", "primal") else x["dTO"])
    res = _run(x, mode)
    for n, t in res.items():
        if n in ref and n not in ("lse", "mu", "li"):
            err = orc.rel_frobenius(t, ref[n])
            assert err <= BOUND[dtype], (n, err)  # (also false for NaN)
    cf = orc.attention_jvp_closed_form(*[x[n] for n in ORDER])
    assert torch.allclose(res["lse"][..., :Lq].double(), torch.as_tensor(cf["lse"]).double(), rtol=2e-5, atol=2e-5)
    assert torch.allclose(res["lse"][..., Lq:], torch.full_like(res["lse"][..., Lq:], Lk).log(), rtol=1e-6)
    if "li" in res:
        assert torch.allclose(res["li"][..., :Lq].double(), torch.as_tensor(cf["li"]).double(), rtol=1e-4)
        assert (res["li"][..., Lq:] == Lk).all() and (res["mu"][..., Lq:] == 0).all()


@pytest.mark.parametrize("D", [64, 36])
def test_parts_whose_keys_all_score_minus_infinity(D):
    """Keys that score -inf against every query (their products overflow) from the second stage on, or everywhere but
    there: without them the results are those of the other keys alone, whichever waves walk them."""
    H, Lq, Lk = 2, 70, 256
    for lost in (slice(32, 256), slice(64, 96), slice(32, 160)):
        x = orc.make_inputs(1, H, Lq, Lk, D, seed=1, tangent_scale=0.3, dtype=torch.bfloat16)
        x["q"][..., 0] = 1.0
        x["k"][..., lost, 0] = -3.0e38
        x["k"][..., lost, 1:] = 0
        x["q"][..., 1] = 1.0
        x["k"][..., lost, 1] = -3.0e38
        x["tq"][..., :2] = 0
        keep = torch.ones(Lk, dtype=torch.bool)
        keep[lost] = False
        part = {n: t[..., keep, :] if n in ("k", "v", "tk", "tv") else t for n, t in x.items()}
        res = _run(x, "both")
        ref = orc.attention_jvp_autograd(*[part[n] for n in ORDER], dO=x["dO"], dTO=x["dTO"])
        for n in ("O", "TO"):
            assert orc.rel_frobenius(res[n], ref[n]) <= 1e-2, (lost, n)


def test_parts_do_what_whole_workgroups_do():
    """The same heads alone and among so many that no launch splits."""
    from semicat_amd import kernels as K
    H, L, D = 300, 384, 64
    gen = torch.Generator(device="cuda").manual_seed(0)
    x = {n: torch.randn((1, H, L, D), device="cuda", generator=gen).bfloat16() for n in (*ORDER, "dO", "dTO")}
    all_ = _run({n: t.cpu() for n, t in x.items()}, "both")
    one = _run({n: t[:, 7:9].cpu() for n, t in x.items()}, "both")
    for n, t in one.items():
        # two results that are each rounded to 16 bits on their own way: sqrt(2) of the 2.6e-3 either is off
        assert orc.rel_frobenius(t, all_[n][:, 7:9]) <= 4e-3, n
