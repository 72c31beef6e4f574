"""The fp32 kernels on rows of every length and alignment: no column beyond the head dimension takes part, whatever lies there,
nothing outside the tensors is written, and rows that no 16-byte boundary fits cost what others of the class cost."""
import pytest
import torch

from oracle import attn_jvp_oracle as orc

pytestmark = pytest.mark.gpu
GRADS = ("dq", "dk", "dv", "dtq", "dtk", "dtv")
TOL = 1e-5  # the bound that the fp32 mode is held to elsewhere


def _gapped(t, gap, offset):
    """A copy of t whose rows are `gap` elements apart, NaN between them, in front and behind."""
    B, H, L, D = t.shape
    buf = torch.full((B * H * L * (D + gap) + offset + 8,), float("nan"), device="cuda")
    v = buf[offset:offset + B * H * L * (D + gap)].view(B, H, L, D + gap)[..., :D]
    v.copy_(t)
    return v, buf


@pytest.mark.parametrize("first", [16, 32, 48, 64, 80, 96, 112, 128])
def test_every_head_dimension_among_nan(first):
    from semicat_amd import kernels as K
    for D in range(first, min(first + 16, 129)):
        gap, offset = 1 + D % 5, D % 3
        x = orc.make_inputs(1, 2, 19, 37, D, seed=D, tangent_scale=0.5, dtype=torch.float32)
        ref = orc.attention_jvp_autograd(*[x[n] for n in orc.TENSOR_ORDER])
        print(f"[f32 rows] D={D} gap={gap} offset={offset}", flush=True)
        d = {n: _gapped(t, gap, offset)[0] for n, t in x.items()}
        out = [_gapped(x["q"], gap, offset) for _ in range(2)]
        g = [_gapped(x[n], gap, offset) for n in ("q", "k", "v", "tq", "tk", "tv")]
        o, to, lse, mu, _ = K.attention_jvp_forward(*[d[n] for n in ("q", "k", "v", "tq", "tk", "tv")], o=out[0][0],
                                                    to=out[1][0])
        K.attention_jvp_backward(*[d[n] for n in ("q", "k", "v", "tq", "tk", "tv")], o, to, lse, mu, dO=d["dO"],
                                 dTO=d["dTO"], grads=tuple(v for v, _ in g))
        for n, t in {"O": o, "TO": to, **{n: v for n, (v, _) in zip(GRADS, g)}}.items():
            err = orc.rel_frobenius(t.cpu(), ref[n])
            assert err <= TOL, (D, n, err)  # (also false for NaN)
        for v, buf in out + g:
            assert buf.isnan().sum() == buf.numel() - v.numel(), D


@pytest.mark.parametrize("D,offset,like", [(65, 0, 68), (127, 0, 128), (64, 1, 64), (35, 0, 36)])
def test_unaligned_rows_cost_what_aligned_rows_cost(D, offset, like):
    from semicat_amd import kernels as K

    def launches(D, offset):
        B, H, L = 64, 12, 128
        make = lambda: torch.randn(B * H * L * D + offset, device="cuda")[offset:].view(B, H, L, D)
        x = [make() for _ in range(8)]
        fwd, (o, to, lse, mu, _) = K.plan_forward(*x[:6], with_li=False)
        fwd()
        bwd, _ = K.plan_backward(*x[:6], o, to, lse, mu, dO=x[6], dTO=x[7])
        return fwd, bwd

    both, best = [launches(D, offset), launches(like, 0)], [float("inf")] * 2
    for _ in range(8):  # in turn, so that clocks and neighbours meet both
        for i, (fwd, bwd) in enumerate(both):
            e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
            e[0].record()
            for _ in range(4):
                fwd()
                bwd()
            e[1].record()
            torch.cuda.synchronize()
            best[i] = min(best[i], e[0].elapsed_time(e[1]) * 250)
    print(f"[f32 rows] D={D}+{offset} {best[0]:.0f} us, D={like} {best[1]:.0f} us")
    assert best[0] < 1.25 * best[1]
