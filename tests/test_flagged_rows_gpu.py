"""The second pass of the row-owned kernel reaches single sharp rows wherever they lie: each form of the first pass writes its part
of the flags of 64 rows (a byte or two each where waves share a group of rows, two words where a wave owns 32)."""
import pytest
import torch

from oracle import attn_jvp_oracle as orc

pytestmark = pytest.mark.gpu
ORDER = ("q", "k", "v", "tq", "tk", "tv")
# One sharp row in every third head: in each group of 16 of the first 64 rows, in later words, in the last rows.
ROWS = (20, 50, 70, 120, 199, 5, 33, 131)


def _inputs(H, Lq, Lk, D, dtype, cot, seed=7):
    x = orc.make_inputs(1, H, Lq, Lk, D, seed=seed, tangent_scale=0.3, dtype=dtype)
    sharp = [(h, ROWS[i % len(ROWS)]) for i, h in enumerate(range(1, H, 3))][:24]
    for h, r in sharp:  # a logit of 10 against its key: 0.97 to 0.99 of the probability
        q = x["q"][0, h, r].float()
        x["k"][0, h, (5 * r) % Lk] = (q * (10 * D ** 0.5 / q.dot(q))).to(dtype)
    if cot == "dO":
        x["dTO"].zero_()
    return x, sharp


def _rows(t, sharp):
    """The sharp rows alone, each by its own norm in the reference."""
    return torch.stack([torch.as_tensor(t)[0, i, r].double() for i, (_, r) in enumerate(sharp)])


def _errors(got, ref):
    return (got - ref).norm(dim=-1) / ref.norm(dim=-1)


def _flagged(x, sharp, dtype):
    """Rows that the kernel's rule certainly flags: a residue of the row sums above the unit roundoff times the row's absolute
    sum, which the kernel samples on every fourth key (at a row with half of it on one key up to 2.5 times the sum)."""
    q, k, v, tq, tk, tv, dO, G = (x[n].double() for n in orc.TENSOR_ORDER)
    s = q.shape[-1] ** -0.5
    P = (s * q @ k.mT).softmax(-1)
    TS = s * (tq @ k.mT + q @ tk.mT)
    N = TS - (P * TS).sum(-1, keepdim=True)
    O, TO = ((P @ v).to(dtype).double(), ((P * N) @ v + P @ tv).to(dtype).double())
    dTS = P * (G @ v.mT - (G * O).sum(-1, keepdim=True))
    dS = dTS * N + P * (G @ tv.mT + dO @ v.mT - (G * TO).sum(-1, keepdim=True) - (dO * O).sum(-1, keepdim=True))
    tau = 2.0 ** (-11 if dtype == torch.float16 else -8)
    over = [(t.sum(-1).abs() > 4 * tau * t.abs().sum(-1))[..., None] for t in (dTS, dS)]
    return _rows(over[0] | over[1], sharp)[:, 0].bool()


# (heads, Lq, Lk, D, type, cotangents): four waves to a group, two, two on rows of odd lengths, 32 rows a wave, one group a wave
@pytest.mark.parametrize("H,Lq,Lk,D,dtype,cot", [(8, 200, 160, 64, torch.bfloat16, "both"), (8, 200, 160, 48, torch.float16, "both"),
                                                 (24, 200, 160, 64, torch.bfloat16, "both"), (16, 200, 160, 36, torch.bfloat16, "both"),
                                                 (171, 257, 260, 64, torch.bfloat16, "dO"), (171, 257, 260, 128, torch.float16, "dO"),
                                                 (64, 200, 160, 64, torch.bfloat16, "both"), (24, 200, 160, 80, torch.float16, "both")])
def test_single_sharp_rows_are_repaired(H, Lq, Lk, D, dtype, cot):
    from semicat_amd import kernels as K
    print(f"[flags] {H} {Lq} {Lk} {D} {dtype} {cot}", flush=True)
    x, sharp = _inputs(H, Lq, Lk, D, dtype, cot)
    d = {n: t.cuda() for n, t in x.items()}
    o, to, lse, mu, _ = K.attention_jvp_forward(*[d[n] for n in ORDER])

    def backward(mode):
        was = K.set_row_sum_repair(mode)
        try:
            return K.attention_jvp_backward(*[d[n] for n in ORDER], o, to, lse, mu, dO=d["dO"], dTO=d["dTO"] if cot == "both" else None)
        finally:
            K.set_row_sum_repair(was)

    auto, off = backward("auto"), backward("off")
    heads = [h for h, _ in sharp]
    one = {n: t[:, heads] for n, t in x.items()}
    args = [one[n] for n in orc.TENSOR_ORDER]
    flagged = _flagged(one, sharp, dtype)
    assert 2 * flagged.sum() > len(sharp)
    ref = orc.attention_jvp_autograd(*args)
    unrepaired = orc.row_sum_rounding_model(*args, dtype=dtype)
    repaired = orc.row_sum_rounding_model(*args, dtype=dtype, repaired=True)
    for name, got, without in (("dq", auto[0], off[0]), ("dtq", auto[3], off[3]))[:2 if cot == "both" else 1]:
        want = _rows(ref[name], sharp)[flagged]
        rows = lambda t: _rows(t, sharp)[flagged]
        bound = 1.5 * _errors(rows(repaired[name]), want).max() + 1e-3  # as for whole tensors of such rows
        assert (_errors(rows(unrepaired[name]), want) > 2 * bound).any()  # the case fails without the repair
        e, e0 = (_errors(rows(t.cpu()[:, heads]), want) for t in (got, without))
        print(name, f"bound {bound:.2e} repaired {e.max():.2e} without {e0.max():.2e}, {len(want)} of {len(sharp)} rows", flush=True)
        assert (e <= bound).all() and (e0 > bound).any(), (name, e, e0)
