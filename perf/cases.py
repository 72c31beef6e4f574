"""The work that is timed: attention-JVP calls and the training step around them, through the package's
public entry points.

A case is a plain dict.  ``kind`` selects the path:

* ``op``      one forward (``attention_jvp_forward``) and one backward (``attention_jvp_backward``) on
              ``[B,H,L,D]`` tensors, as a program with its own autograd glue calls them.  ``cot`` says which
              outputs have a cotangent, ``seq_major`` whether the tensors are views of ``[B,L,H,D]`` memory.
* ``primal``  the same without tangents: plain attention and its backward.
* ``autograd``  ``safe_sdpa_jvp`` on ``[B,S,H,D]`` tensors under ``torch.func.jvp``, then the gradients of
              all six inputs by reverse mode: how a network's forward-mode step reaches the op.
* ``rotary``  ``safe_sdpa_jvp_rotary`` on q, k, v views of one fused projection, under ``torch.func.jvp``, then
              the gradients of the projection and its tangent.
* ``train``   both losses of the training step on the DiT under bf16 autocast, and their backward.

Flop counts are those of the contractions alone: 6 of them (12 without the factor 2) per (query, key, column)
forward with tangents, 15 backward with both cotangents, 2 and 5 without tangents.
"""
import math

import torch

from semicat_amd import (attention_forward, attention_jvp_backward, attention_jvp_forward, safe_sdpa_jvp,
                         safe_sdpa_jvp_rotary)
from semicat_amd import train_step
from semicat_amd.dit import DIT, Rotary

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
SIZES = {"bf16": 2, "fp16": 2, "fp32": 4}
DEVICE = "cuda"


def _op(name, B, H, Lq, Lk, D, dtype, cot="both", seq_major=False):
    return {"name": name, "kind": "op", "B": B, "H": H, "Lq": Lq, "Lk": Lk, "D": D, "dtype": dtype, "cot": cot,
            "seq_major": seq_major}


def listed():
    return [
        # The smallest of the shapes that the op is tested on against the eager math path: a call of a toy model,
        # all launches and host time.
        _op("toy_fp16", 2, 2, 16, 16, 32, "fp16"),
        # One fp32 call of a small model at full fp32 precision (the correctness configuration).
        _op("fp32_config", 2, 4, 256, 256, 64, "fp32"),
        # The attention of the LM1B DiT at batch 64 with a tangent on every sample: the headline workload.
        _op("lm1b_bf16", 64, 12, 128, 128, 64, "bf16"),
        # The character-level (text8) DiT: twice the batch, twice the sequence.
        _op("text8_bf16", 128, 12, 256, 256, 64, "bf16"),
        # The middle of the long-sequence sweep.
        _op("long_1024_d64_bf16", 8, 16, 1024, 1024, 64, "bf16"),
        # Its largest point: the longest sequence at the widest head.
        _op("long_4096_d128_bf16", 8, 16, 4096, 4096, 128, "bf16"),
        # Cross attention between ragged sequences in the caller's [B,L,H,D] layout, reverse mode through the
        # tangent output only.
        _op("ragged_cross_fp16", 4, 6, 333, 205, 48, "fp16", cot="dTO", seq_major=True),
        # A head dimension that leaves rows without 16-byte alignment.
        _op("odd_head_bf16", 8, 8, 300, 300, 36, "bf16"),
        # Plain attention (the samples of a batch without tangents, and sampling's forward) and its backward.
        {"name": "primal_1024_bf16", "kind": "primal", "B": 8, "H": 16, "Lq": 1024, "Lk": 1024, "D": 64,
         "dtype": "bf16"},
        # A network in fp32 without autocast: the op computes in bf16 and hands fp32 back.
        {"name": "lm1b_fp32_callers", "kind": "autograd", "B": 64, "H": 12, "S": 128, "D": 64, "dtype": "fp32"},
        # One block's attention of the self-distillation share (a quarter of 64 samples) with its rotary embedding.
        {"name": "lm1b_rotary_block", "kind": "rotary", "B": 16, "H": 12, "S": 128, "D": 64, "dtype": "bf16"},
        # The training step of the LM1B DiT: cross-entropy on 48 samples, self-distillation through forward-mode
        # AD on 16.
        {"name": "lm1b_train_step", "kind": "train", "B": 64, "split": 16, "S": 128, "H": 12, "V": 30522,
         "blocks": 12},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cost(c):
    """Time of the case at the rates the kernels reach, in arbitrary units, to keep drawn cases affordable."""
    slow = 12.0 if c["dtype"] == "fp32" else 1.0
    pad = 32 if c["D"] <= 32 else 64 if c["D"] <= 64 else 128
    return slow * c["B"] * c["H"] * c["Lq"] * c["Lk"] * pad


def draw(rng):
    kind = rng.choice(("op", "op", "op", "op", "op", "primal", "autograd", "rotary", "train"))
    if kind == "train":
        # the character vocabulary or the word-piece one, batches from one accumulation slice to the whole step
        text8 = rng.random() < 0.5
        B = rng.randint(8, 64)
        return {"kind": "train", "B": B, "split": max(1, B // 4), "S": rng.choice((64, 128)), "H": 12,
                "V": 27 if text8 else rng.randint(8000, 30522), "blocks": rng.randint(2, 12)}
    if kind == "autograd":
        return {"kind": kind, "B": _log_int(rng, 2, 64), "H": rng.choice((4, 8, 12, 16)), "S": _log_int(rng, 32, 512),
                "D": rng.choice((32, 64, 64, 128)), "dtype": rng.choice(("fp32", "fp32", "bf16"))}
    if kind == "rotary":
        return {"kind": kind, "B": _log_int(rng, 4, 64), "H": rng.choice((8, 12, 16)), "S": _log_int(rng, 64, 1024),
                "D": rng.choice((64, 64, 128)), "dtype": "bf16"}
    most = _cost(listed()[5])
    while True:
        dtype = rng.choice(("bf16", "bf16", "fp16", "fp32")) if kind == "op" else rng.choice(("bf16", "fp16"))
        Lq = _log_int(rng, 8, 4096)
        Lk = Lq if rng.random() < 0.7 else _log_int(rng, 8, 4096)
        c = {"kind": kind, "B": _log_int(rng, 1, 128), "H": rng.randint(1, 16), "Lq": Lq, "Lk": Lk,
             "D": rng.choice((16, 20, 32, 36, 48, 64, 64, 64, 80, 128, 128)), "dtype": dtype}
        if kind == "op":
            c["cot"] = rng.choice(("both", "both", "both", "dTO", "dO"))
            c["seq_major"] = rng.random() < 0.4
        if _cost(c) <= 0.5 * most and c["B"] * c["H"] * max(Lq, Lk) * c["D"] <= 1 << 27:
            return c


def _randn(gen, shape, scale, dtype):
    return (torch.randn(shape, device=DEVICE, generator=gen) * scale).to(dtype)


def prepare(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    kind = case["kind"]
    if kind == "train":
        return _prepare_train(case, seed, gen)
    B, H, D, dt = case["B"], case["H"], case["D"], DTYPES[case["dtype"]]
    if kind in ("op", "primal"):
        Lq, Lk = case["Lq"], case["Lk"]

        def make(L, scale):
            if case.get("seq_major"):
                return _randn(gen, (B, L, H, D), scale, dt).transpose(1, 2)
            return _randn(gen, (B, H, L, D), scale, dt)

        s = {"q": make(Lq, 1.0), "k": make(Lk, 1.0), "v": make(Lk, 1.0)}
        if kind == "op":
            s.update(tq=make(Lq, 0.1), tk=make(Lk, 0.1), tv=make(Lk, 0.1))
        if case.get("cot", "dO") in ("both", "dO"):
            s["dO"] = make(Lq, 1.0)
        if case.get("cot", "dO") in ("both", "dTO"):
            s["dTO"] = make(Lq, 1.0)
        return {"kind": kind, **s}
    S = case["S"]
    if kind == "autograd":
        x = [_randn(gen, (B, S, H, D), scale, dt).requires_grad_() for scale in (1.0, 1.0, 1.0, 0.1, 0.1, 0.1)]
        return {"kind": kind, "x": x, "g": [_randn(gen, (B, S, H, D), 1.0, dt) for _ in range(2)]}
    cos, sin = Rotary(S, D).to(DEVICE).half_tables()
    qkv = _randn(gen, (B, S, 3, H, D), 1.0, dt).requires_grad_()
    tqkv = _randn(gen, (B, S, 3, H, D), 0.1, dt).requires_grad_()
    return {"kind": kind, "qkv": qkv, "tqkv": tqkv, "cos": cos, "sin": sin,
            "g": [_randn(gen, (B, S, H, D), 1.0, dt) for _ in range(2)]}


def _prepare_train(case, seed, gen):
    B, S, V = case["B"], case["S"], case["V"]
    torch.manual_seed(seed)
    with torch.device(DEVICE):
        net = DIT(vocab_size=V, hidden_size=64 * case["H"], cond_dim=128, n_blocks=case["blocks"], n_heads=case["H"],
                  dropout=0.0, length=S)
        for p in net.parameters():
            # the layers that start at zero hide everything in front of them from the gradients: a step in the
            # middle of training has them away from zero
            torch.nn.init.normal_(p, std=0.02)
        for m in net.modules():
            if isinstance(m, torch.nn.LayerNorm):
                m.weight.data.add_(1.0)
    # One bucket that holds every gradient, in it the same layer of all blocks side by side.
    groups = {}
    for name, p in net.named_parameters():
        parts = name.split(".")
        groups.setdefault(".".join(parts[2:]) if parts[0] == "blocks" else name, []).append(p)
    flat = torch.zeros(sum(p.numel() for p in net.parameters()), device=DEVICE)
    grads, at = {}, 0
    for name, params in groups.items():
        start = at
        for p in params:
            p.grad = flat[at:at + p.numel()].view_as(p)
            at += p.numel()
        grads[name] = flat[start:at]
    t = torch.rand(B, device=DEVICE, generator=gen)
    return {"kind": "train", "net": net, "flat": flat, "grads": grads, "split": case["split"],
            "x0": torch.randn((B, S, V), device=DEVICE, generator=gen),
            "x1": torch.randint(0, V, (B, S), device=DEVICE, generator=gen),
            "t": t, "s": t * torch.rand(B, device=DEVICE, generator=gen)}


def run(state):
    return RUN[state["kind"]](state)


def _run_op(s):
    o, to, lse, mu, _ = attention_jvp_forward(s["q"], s["k"], s["v"], s["tq"], s["tk"], s["tv"], with_li=False)
    grads = attention_jvp_backward(s["q"], s["k"], s["v"], s["tq"], s["tk"], s["tv"], o, to, lse, mu,
                                   dO=s.get("dO"), dTO=s.get("dTO"))
    return o, to, lse, mu, grads


def _run_primal(s):
    o, lse = attention_forward(s["q"], s["k"], s["v"])
    grads = attention_jvp_backward(s["q"], s["k"], s["v"], None, None, None, o, None, lse, None, dO=s["dO"])
    return o, lse, grads


def _run_autograd(s):
    q, k, v, tq, tk, tv = s["x"]
    y, ty = torch.func.jvp(safe_sdpa_jvp, (q, k, v), (tq, tk, tv))
    return y, ty, torch.autograd.grad((y, ty), s["x"], s["g"])


def _run_rotary(s):
    def attend(qkv):
        return safe_sdpa_jvp_rotary(qkv[:, :, 0], qkv[:, :, 1], qkv[:, :, 2], s["cos"], s["sin"])

    y, ty = torch.func.jvp(attend, (s["qkv"],), (s["tqkv"],))
    return y, ty, torch.autograd.grad((y, ty), (s["qkv"], s["tqkv"]), s["g"])


def _run_train(s):
    n, x0, x1, t = s["split"], s["x0"], s["x1"], s["t"]
    s["flat"].zero_()
    with torch.autocast(device_type=DEVICE, dtype=torch.bfloat16):
        vf = train_step.vfm_loss(s["net"], x0[n:], x1[n:], t=t[n:])
        sd = train_step.lag_self_distillation_loss(s["net"], x0[:n], x1[:n], t=t[:n], s=s["s"][:n])
    (vf + sd).backward()
    return vf.detach(), sd.detach(), s["grads"]


RUN = {"op": _run_op, "primal": _run_primal, "autograd": _run_autograd, "rotary": _run_rotary, "train": _run_train}


def work(case):
    kind = case["kind"]
    if kind == "train":
        B, S, V, W = case["B"], case["S"], case["V"], 64 * case["H"]
        n = case["split"]
        per_block = 12 * W * W + 6 * 128 * W
        params = case["blocks"] * per_block + 2 * W * V
        attention = case["blocks"] * S * S * W  # (query, key, column) triples of one sample
        # matrix products: cross-entropy share forward + backward (3 passes of 2 flops per weight and token, 14 per
        # triple), self-distillation share with tangents (primal and tangent forward, both directions back) and its
        # target network (one forward)
        flops = (B - n) * (6 * S * params + 14 * attention) + n * (14 * S * params + 46 * attention)
        # x0 once, every parameter and its gradient once
        return {"bytes": 4 * B * S * V + 8 * params, "flops": flops}
    B, H, D, e = case["B"], case["H"], case["D"], SIZES[case["dtype"]]
    if kind in ("op", "primal"):
        Lq, Lk = case["Lq"], case["Lk"]
        triples = B * H * Lq * Lk * D
        rows_q, rows_k = B * H * Lq * D * e, B * H * Lk * D * e
        cot = case.get("cot", "dO")
        if kind == "primal":
            # read q, k, v, dO; write o, dq, dk, dv
            return {"bytes": 4 * rows_q + 4 * rows_k, "flops": 14 * triples}
        tangent = cot != "dO"
        n_cot = 2 if cot == "both" else 1
        # read the six inputs and the cotangents, write o, to and the gradients
        by = rows_q * (2 + 2 + n_cot + (2 if tangent else 1)) + rows_k * (4 + (4 if tangent else 2))
        return {"bytes": by, "flops": (12 + {"both": 30, "dTO": 26, "dO": 10}[cot]) * triples}
    S = case["S"]
    # read six inputs (or the two projections) and two cotangents, write two outputs and six gradients
    return {"bytes": 16 * B * H * S * D * e, "flops": 42 * B * H * S * S * D}


def tolerance(case):
    """Four times what was measured, over the listed shapes and forty drawn ones, against the same formulas in
    fp64: bf16 2.6e-3 (largest single difference 2.9e-2 of the root mean square or of the value), fp16 3.3e-4
    (4.0e-3), fp32 1.3e-6 (1.2e-5).  The training step's gradients go through twelve blocks of bf16 products:
    with eager attention in bf16 in place of the op they differ by 1.2e-2 (0.30), with every layer in fp32 by
    1.4e-2 (0.34)."""
    if case["kind"] == "train":
        return {"rel": 3e-2, "max": 0.9}
    if case["dtype"] == "fp16":
        return {"rel": 1.3e-3, "max": 1.6e-2}
    if case["kind"] == "op" and case["dtype"] == "fp32":
        return {"rel": 5e-6, "max": 5e-5}
    return {"rel": 1e-2, "max": 0.12}
