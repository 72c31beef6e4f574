"""The column-owned launch computes the same whatever comes with it: repair on or off, with the row-owned launch or in a call of its
own."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# (heads, Lq, Lk, D): two and four waves to a group of keys, rows of odd lengths, whole workgroups, 32 keys a wave
@pytest.mark.parametrize("H,Lq,Lk,D,dtype", [(8, 160, 256, 64, torch.bfloat16), (24, 130, 257, 48, torch.float16), (2, 400, 300, 36, torch.bfloat16),
                                             (30, 200, 513, 64, torch.bfloat16), (9, 77, 150, 128, torch.float16), (260, 513, 257, 32, torch.bfloat16)])
@pytest.mark.parametrize("cot", ["both", "dO", "dTO"])
def test_same_bits(H, Lq, Lk, D, dtype, cot):
    from semicat_amd import _lib, kernels as K
    print(f"[modes] {H} {Lq} {Lk} {D} {dtype} {cot}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(Lq + D)

    def rand(L, scale=1.0):
        return (torch.randn((1, H, L, D), device="cuda", generator=gen) * scale).to(dtype)

    x = [rand(Lq), rand(Lk), rand(Lk), rand(Lq, 0.1), rand(Lk, 0.1), rand(Lk, 0.1)]
    o, to, lse, mu, _ = K.attention_jvp_forward(*x)
    cots = {n: rand(Lq) for n in (("dO", "dTO") if cot == "both" else (cot,))}
    columns = (1, 2) if cot == "dO" else (1, 2, 4, 5)

    def backward(**kw):
        return K.attention_jvp_backward(*x, o, to, lse, mu, **cots, **kw)

    ref = backward()
    was = K.set_row_sum_repair("off")
    try:
        off = backward()
    finally:
        K.set_row_sum_repair(was)
    workspace = torch.zeros(_lib.load().sjvp_bwd_workspace_bytes(1, H, Lq, Lk, D, _lib.SJVP_BF16), device="cuda", dtype=torch.uint8)
    grads = tuple(None if g is None else torch.empty_like(g) for g in ref)
    for part in (_lib.SJVP_BWD_ROW, _lib.SJVP_BWD_COL):
        backward(grads=grads, workspace=workspace, parts=part)
    assert all(torch.equal(grads[i], ref[i]) for i in columns)
    assert all(torch.equal(off[i], ref[i]) for i in columns)
