"""The fp32 kernels that take their operands in three bf16 parts, at the edges of their tiles, workgroups and head-dimension
classes, against the fp64 oracle; and heads that hold numbers for the fp32 unit, against the same heads in a call that the fp32
unit's kernels serve as a whole."""
import pytest
import torch
from torch.profiler import ProfilerActivity, profile

from oracle import attn_jvp_oracle as orc

pytestmark = pytest.mark.gpu
NAMES = ("o", "to", "lse", "mu", "dq", "dk", "dv", "dtq", "dtk", "dtv")
TOL = 1e-5  # the bound that the fp32 mode is held to elsewhere


def _step(x, mode="both"):
    from semicat_amd import kernels as K
    ins = [x[n] for n in ("q", "k", "v", "tq", "tk", "tv")]
    o, to, lse, mu, _ = K.attention_jvp_forward(*ins, with_li=False)
    if mode == "dO":
        ins[3:] = [None] * 3
    g = K.attention_jvp_backward(*ins, o, None if mode == "dO" else to, lse, None if mode == "dO" else mu,
                                 dO=None if mode == "dTO" else x["dO"], dTO=None if mode == "dO" else x["dTO"])
    return dict(zip(NAMES, (o, to, lse, mu, *g)))


def _kernels(run):
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        res = run()
        torch.cuda.synchronize()
    return res, [e.key for e in prof.key_averages() if "f32" in e.key]


@pytest.mark.parametrize("mode", ["both", "dO", "dTO"])
@pytest.mark.parametrize("B,H,Lq,Lk,D,offset", [
    (40, 12, 75, 90, 64, 0),   # eight waves, ragged rows and last stage; waves and a workgroup's half without rows
    (25, 4, 100, 97, 64, 1),   # four waves, a last stage of one row, no 16-byte alignment
    (30, 12, 129, 100, 48, 0),  # a second workgroup with one row
    (40, 12, 96, 127, 33, 3),  # odd columns
    (30, 12, 100, 120, 32, 0), (30, 12, 100, 120, 21, 1), (30, 12, 80, 96, 16, 0),
    (20, 12, 90, 90, 80, 0), (20, 12, 90, 95, 67, 2), (16, 12, 100, 100, 128, 0), (20, 12, 120, 110, 101, 1)])
def test_parts_at_the_edges(mode, B, H, Lq, Lk, D, offset):
    x = orc.make_inputs(B, H, Lq, Lk, D, seed=7, tangent_scale=0.5, dtype=torch.float32)
    cot = {n: x[n] for n in ("dO", "dTO") if mode in ("both", n)}
    ref = orc.attention_jvp_autograd(*[x[n] for n in orc.TENSOR_ORDER[:6]], **cot)
    d = {}
    for n, t in x.items():  # views that start `offset` elements into their storage, in [B,L,H,D] memory
        buf = torch.empty(t.numel() + offset, device="cuda")
        d[n] = buf[offset:].view(B, t.shape[2], H, D).transpose(1, 2)
        d[n].copy_(t)
    print(f"[f32 parts] {(B, H, Lq, Lk, D, offset)} {mode}", flush=True)
    res, names = _kernels(lambda: _step(d, mode))
    assert any("fwd_f32x3" in n for n in names) and any("row_f32x3" in n for n in names), names
    assert any("col_f32x3" in n for n in names), names
    for n, t in res.items():
        if t is not None and n not in ("lse", "mu"):
            err = orc.rel_frobenius(t.cpu(), ref[n.upper() if n in ("o", "to") else n])
            assert err <= TOL, (n, err)
    assert (res["lse"][..., Lq:] - torch.tensor(float(Lk)).log().item()).abs().max() <= 1e-5
    assert not res["mu"][..., Lq:].any()
    from semicat_amd import kernels as K
    o, lse = K.attention_forward(d["q"], d["k"], d["v"])
    assert orc.rel_frobenius(o.cpu(), ref["O"]) <= TOL and torch.allclose(lse, res["lse"], rtol=1e-6, atol=1e-6)


@pytest.mark.parametrize("B,H,Lq,Lk,D,parts", [(16, 16, 200, 32, 100, True), (83, 3, 172, 172, 128, True), (15, 8, 76, 76, 80, True),
                                              (30, 12, 100, 120, 64, True), (12, 16, 200, 500, 80, True), (13, 6, 52, 700, 20, False),
                                              (36, 4, 144, 144, 64, True)])
def test_one_set_for_a_forward_with_tangents_and_a_cotangent_on_o(B, H, Lq, Lk, D, parts):
    """The backward knows no tangents there.  Mixed with the other set's forward its error is 1.1 to 1.2 times the fp32 unit's."""
    x = orc.make_inputs(B, H, Lq, Lk, D, seed=7, tangent_scale=0.1, dtype=torch.float32)
    ref = orc.attention_jvp_autograd(*[x[n] for n in orc.TENSOR_ORDER[:6]], dO=x["dO"])
    d = {n: t.cuda() for n, t in x.items()}
    print(f"[f32 one set] {(B, H, Lq, Lk, D)}", flush=True)
    res, names = _kernels(lambda: _step(d, "dO"))
    assert len(names) == 3 and all(("f32x3" in n) == parts for n in names), names
    _, names = _kernels(lambda: _step(d, "both"))
    assert len(names) == 3 and all(("f32x3" in n) == parts for n in names), names
    # calls of one batch element are too small for the other set, and split groups of rows: the smallest error the unit's kernels have
    unit = [_step({n: t[b:b + 1] for n, t in d.items()}, "dO") for b in range(B)] if parts else []
    for n in ("o", "to", "dq", "dk", "dv") if parts else ():
        r = ref[n.upper() if n in ("o", "to") else n]
        err, unit_err = (orc.rel_frobenius(t.cpu(), r) for t in (res[n], torch.cat([u[n] for u in unit])))
        print(f"  {n} {err:.3e} {unit_err:.3e}")
        assert err <= 1.02 * unit_err, (n, err, unit_err)


@pytest.mark.parametrize("mode", ["both", "dTO", "plain"])
@pytest.mark.parametrize("B,H,Lq,Lk,D", [(30, 12, 100, 120, 64), (24, 8, 160, 600, 64), (24, 12, 520, 70, 64), (40, 12, 75, 90, 48),
                                        (30, 12, 100, 120, 16), (12, 16, 200, 500, 80), (32, 4, 300, 520, 128)])
def test_error_is_not_above_the_units(mode, B, H, Lq, Lk, D):
    """Every output against fp64, beside the same heads in calls that the fp32 unit serves (split groups: its smallest error)."""
    from semicat_amd import kernels as K
    x = orc.make_inputs(B, H, Lq, Lk, D, seed=11, tangent_scale=0.5, dtype=torch.float32)
    cot = {n: x[n] for n in ("dO", "dTO") if n in {"both": ("dO", "dTO"), "dTO": ("dTO",), "plain": ("dO",)}[mode]}
    ref = orc.attention_jvp_autograd(*[x[n] for n in orc.TENSOR_ORDER[:6]], **cot)
    d = {n: t.cuda() for n, t in x.items()}

    def step(y):
        if mode != "plain":
            return _step(y, mode)
        o, lse = K.attention_forward(y["q"], y["k"], y["v"])
        g = K.attention_jvp_backward(y["q"], y["k"], y["v"], None, None, None, o, None, lse, None, dO=y["dO"])
        return {"o": o, **dict(zip(("dq", "dk", "dv"), g))}

    print(f"[f32 error] {(B, H, Lq, Lk, D)} {mode}", flush=True)
    res, names = _kernels(lambda: step(d))
    assert len(names) == 3 and all("f32x3" in n for n in names), names
    unit, names = _kernels(lambda: [step({n: t[b:b + 1] for n, t in d.items()}) for b in range(B)])
    assert not any("f32x3" in n for n in names), names
    for n in ("o", "to", "dq", "dk", "dv", "dtq", "dtk", "dtv"):
        if res.get(n) is not None:
            r = ref[n.upper() if n in ("o", "to") else n]
            err, unit_err = (orc.rel_frobenius(t.cpu(), r) for t in (res[n], torch.cat([u[n] for u in unit])))
            print(f"  {n} {err:.3e} {unit_err:.3e}")
            assert err <= 1.02 * unit_err, (n, err, unit_err)


def _at(name, row, value, column=0):
    def put(x, b):
        x[name][b, 0, row, column] = value
    return put


def _overflowing(x, b):  # one score beyond the range
    for n in ("q", "k", "tq", "tk"):
        x[n][b, 0, :, 0] = 0.0
    x["q"][b, 0, 5, 0], x["k"][b, 0, 9, 0] = 1e25, -1e25


def _lowest(x, b):
    x["q"][b, 0, :, 0] = 8.0
    x["k"][b, 0, 40:, 0] = torch.finfo(torch.float32).min
    x["tq"][b, 0, :, 0] = x["tk"][b, 0, :, 0] = 0.0


def _tiny_rows(x, b):
    x["dO"][b, 0, 70] *= 2.0 ** -110
    x["tk"][b, 0, 9] *= 2.0 ** -120


SPECIAL = [_at("k", 3, float("inf")), _at("k", 33, float("-inf"), 7), _at("q", 17, float("nan")), _at("v", 40, float("inf"), 20),
           _at("tv", 0, float("-inf")), _at("tk", 8, 1e30), _at("dTO", 11, float("inf"), 3), _at("dO", 70, float("nan"), 31),
           _overflowing, _lowest, _at("v", 2, torch.finfo(torch.float32).max), _at("tq", 1, 1e25), _tiny_rows,
           _at("k", 44, float("nan")), _at("v", 3, float("nan"), 30), _at("tk", 60, float("nan"), 9), _at("dTO", 2, float("nan"))]


@pytest.mark.parametrize("D", [32, 64, 80, 128])
def test_numbers_for_the_fp32_unit(D):
    """They reach the same outputs, as the same infinities and NaN, and no other head."""
    B, L = 480, 75 if D < 80 else 110
    gen = torch.Generator(device="cuda").manual_seed(2)
    x = {n: torch.randn((B, 1, L, D), device="cuda", generator=gen) * (0.5 if n[0] == "t" else 1.0)
         for n in ("q", "k", "v", "tq", "tk", "tv", "dO", "dTO")}
    clean, names = _kernels(lambda: _step(x))
    assert all("f32x3" in n for n in names), names
    heads = [(37 * i + 5) % B for i in range(len(SPECIAL))]
    for b, put in zip(heads, SPECIAL):
        put(x, b)
    print(f"[f32 unit's numbers] D={D}", flush=True)
    got = _step(x)
    unit, names = _kernels(lambda: _step({n: t[heads].contiguous() for n, t in x.items()}))
    assert not any("f32x3" in n for n in names), names
    others = [b for b in range(B) if b not in heads]
    for n in NAMES:
        assert torch.equal(got[n][others], clean[n][others]), n
        a, r = got[n][heads], unit[n]
        for i in range(len(heads)):
            finite = r[i].isfinite()
            assert torch.equal(a[i].isfinite(), finite) and torch.equal(a[i].isnan(), r[i].isnan()), (n, i)
            assert torch.equal(a[i][r[i].isinf()], r[i][r[i].isinf()]), (n, i)
            if finite.any():  # sums of the same products in another order
                assert (a[i][finite] - r[i][finite]).abs().max() <= TOL * r[i][finite].abs().max(), (n, i)


@pytest.mark.parametrize("B,H,Lq,Lk,D", [(30, 12, 100, 120, 64), (30, 8, 120, 100, 32), (16, 12, 100, 100, 128), (30, 4, 75, 90, 48)])
@pytest.mark.parametrize("powers", [{"dO": -118, "dTO": -118}, {"dO": -99, "dTO": -99}, {"v": -60, "tv": -60, "dO": -52, "dTO": -52},
                                    {"tq": -114, "tk": -114, "tv": -114}, {"dTO": -70, "tq": -45, "tk": -45, "tv": -45}])
def test_small_numbers_keep_their_bits(B, H, Lq, Lk, D, powers):
    """Numbers, and products of numbers, below what three bf16 parts hold.  Bound: the error of calls that the fp32 unit serves as a whole, times
    what it grows by against a forward of the other set (1.08 to 1.21) and by sums over the whole axis in the place of four (1.08 to 1.27)."""
    x = orc.make_inputs(B, H, Lq, Lk, D, seed=3, tangent_scale=0.5, dtype=torch.float32)
    x = {n: t * 2.0 ** powers.get(n, 0) for n, t in x.items()}
    ref = orc.attention_jvp_autograd(*[x[n] for n in orc.TENSOR_ORDER[:6]], dO=x["dO"], dTO=x["dTO"])
    d = {n: t.cuda() for n, t in x.items()}
    print(f"[f32 small numbers] {(B, H, Lq, Lk, D)} {powers}", flush=True)
    res, names = _kernels(lambda: _step(d))
    assert all("f32x3" in n for n in names), names
    # calls of one batch element are too small for these kernels
    unit = [_step({n: t[b:b + 1] for n, t in d.items()}) for b in range(B)]
    for n in NAMES:
        if n not in ("lse", "mu"):
            r = ref[n.upper() if n in ("o", "to") else n]
            scale = 2.0 ** -r.abs().max().log2().round().item()  # (its square is beyond fp32, not beyond fp64)
            err, unit_err = (orc.rel_frobenius(t.cpu().double() * scale, r * scale) for t in (res[n], torch.cat([u[n] for u in unit])))
            print(f"  {n} {err:.2e} {unit_err:.2e}")
            assert err <= 1.55 * unit_err, (n, err, unit_err)
