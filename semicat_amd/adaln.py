"""The element-wise parts of the DiT's blocks as single launches (csrc/sjvp_adaln.hip): LayerNorm with adaLN
modulation, the gated residual in front of it, and the MLP's tanh GELU, each with forward-mode tangents and the
reverse mode of both.

As separate PyTorch operations these are what a training step spends its launches on: forward-mode LayerNorm
alone is some twenty kernels and its reverse twice as many, and the step issues thousands of them, each
shorter than the time the host takes to issue it.

The functions serve what a step under bf16 autocast on a GPU has in hand: bf16 activations with fp32 LayerNorm
parameters, outside every transform or inside exactly one ``torch.func.jvp``.  For anything else (other types, other
transforms, tracing, dual numbers, tensor subclasses, modules with hooks) they return None and the caller runs its
PyTorch operations.  To torch.compile they are opaque, like the attention op: a compiled network computes what the
unwrapped one does.  Results are rounded where the PyTorch operations round (the residual stream) or where autocast would
round behind them (the input of the next linear layer).

The reverse mode of the normalised rows' tangent holds the mean and the reciprocal deviation of its input constant: that
is what PyTorch's layer_norm does there, and a network's gradients are the same whichever of the two computes it.  It is
not the full derivative of the tangent."""
from __future__ import annotations

import contextlib
import ctypes
import math
from typing import Optional

import torch
import torch.autograd.forward_ad as fwAD
from torch import Tensor, nn
from torch._C import _functorch
from torch.nn.modules import module as _module

from . import _lib, functional, kernels
from .functional import _below_jvp, _dual_above

_MOD = ("gate", "tgate", "scale", "tscale", "shift", "tshift")
_ARGUMENTS = ("x", "a", "gate", "scale", "shift", "w", "b", "tx", "ta", "tgate", "tscale", "tshift")


def _aligned(t: Optional[Tensor], bytes_: int = 16) -> Optional[Tensor]:
    """The tensor as contiguous memory that starts on a boundary of ``bytes_``."""
    if t is None:
        return None
    t = t.contiguous()
    return t if t.data_ptr() % bytes_ == 0 else t.clone()


def _mod_rows(t: Optional[Tensor]) -> Optional[Tensor]:
    """``[B,1,W]`` with rows of unit stride that start on 8-byte boundaries; the rows of a chunked projection
    are left where they are."""
    if t is None:
        return None
    if t.stride(-1) == 1 and t.stride(0) % 4 == 0 and t.data_ptr() % 8 == 0:
        return t
    return t.contiguous().clone()


def _laid_out(tensors: dict) -> dict:
    """The named tensors as the launches read them; those that are so already are handed back themselves."""
    return {n: _mod_rows(t) if n in _MOD else _aligned(t) for n, t in tensors.items()}


def _outputs(like: Tensor, first: bool = True, second: bool = True, shape=None):
    """Uninitialised memory for an output and its tangent (or either), each with a storage of its own: of a tangent whose
    storage offset or size differs from its primal's, ``make_dual`` keeps a copy in zeroed memory of the whole
    storage's size."""
    shape = like.shape if shape is None else shape
    return tuple(torch.empty(shape, device=like.device, dtype=like.dtype) if wanted else None
                 for wanted in (first, second))


def _pair(like: Tensor, first: bool = True, second: bool = True):
    """Uninitialised memory for the gradients of a tensor and its tangent (or either), side by side, so that the
    reverse mode of a linear layer in front takes both as the rows of one product."""
    both = torch.empty((int(first) + int(second), *like.shape), device=like.device, dtype=like.dtype).unbind(0)
    return (both[0] if first else None), (both[-1] if second else None)


def _stacked(p: Tensor, t: Tensor) -> Tensor:
    """The rows of both tensors as one matrix, without a copy where they lie side by side."""
    rows, W = p.numel() // p.shape[-1], p.shape[-1]
    if torch.is_grad_enabled():  # a recorded backward
        return torch.cat((p.reshape(rows, W), t.reshape(rows, W)))
    p, t = p.detach().contiguous(), t.detach().contiguous()
    if t.data_ptr() == p.data_ptr() + p.numel() * p.element_size() \
            and t.untyped_storage().data_ptr() == p.untyped_storage().data_ptr():
        return p.as_strided((2 * rows, W), (W, 1))
    return torch.cat((p.view(rows, W), t.view(rows, W)))


@torch._dynamo.disable
def _launch(fn, jvp: bool, shape, eps: float, tensors: dict) -> None:
    """Fill the call's structure and launch on the current stream of the tensors' device.  ``tensors`` keeps every
    buffer alive until the launch is queued.  (Through the host extension where it takes the call: 25 us less of host time.)"""
    host = _lib.host()
    status = host.adaln(fn == "sjvp_adaln_bwd", jvp, *shape, eps, tensors) if host else None
    if status is not None:
        return _lib.check(status)
    p = _lib.AdaLn()
    p.B, p.S, p.W = shape
    p.eps = eps
    for name, t in tensors.items():
        if t is not None:
            setattr(p, name, t.data_ptr())
    for i, name in enumerate(_MOD):
        t = tensors.get(name)
        if t is not None:
            p.mod_stride[i] = t.stride(0)
    with torch.cuda.device(tensors["x"].device):
        if fn == "sjvp_adaln_bwd":
            floats = _lib.load().sjvp_adaln_workspace_floats(ctypes.byref(p))
            workspace = torch.empty(floats, device=tensors["x"].device, dtype=torch.float32)
            p.workspace = workspace.data_ptr()
        stream = torch.cuda.current_stream().cuda_stream
        _lib.check(getattr(_lib.load(), fn)(ctypes.byref(p), int(jvp), stream))


def _recorded(outputs, inputs, cotangents):
    """Gradients of ``outputs`` as operations that autograd records: what a backward with ``create_graph`` takes in the
    place of a launch, which has no derivative.  None for an input that needs none."""
    at = [i for i, z in enumerate(inputs) if z is not None and z.requires_grad]
    pairs = [(o, c.to(o.dtype)) for o, c in zip(outputs, cotangents) if c is not None and o.requires_grad]
    grads = [None] * len(inputs)
    if at and pairs:
        found = torch.autograd.grad([o for o, _ in pairs], [inputs[i] for i in at], [c for _, c in pairs],
                                    create_graph=True, allow_unused=True)
        for i, g in zip(at, found):
            grads[i] = g
    return grads


def _plus(*terms):
    """Sum of the terms that are there."""
    terms = [z for z in terms if z is not None]
    return sum(terms[1:], terms[0]) if terms else None


def _times(p, q):
    return None if p is None or q is None else p * q


def _gated_norm_recorded(t: dict, jvp: bool, eps: float, dy, dh, dty, dth) -> dict:
    """The reverse mode of :class:`GatedNormFunction` in recorded PyTorch operations."""
    out = {}
    if t["w"] is not None:
        gated = t["a"] is not None
        y, ty = (t["y"], t["ty"]) if gated else (t["x"], t["tx"])
        w, b, scale, shift, tscale, tshift = (t[n] for n in ("w", "b", "scale", "shift", "tscale", "tshift"))
        y32, scale32 = y.float(), 1.0 + scale.float()
        mean = y32.mean(-1, keepdim=True)
        r = (y32.var(-1, unbiased=False, keepdim=True) + eps).rsqrt()
        normed = (y32 - mean) * r * w + b
        outputs, cotangents = [normed * scale32 + shift.float()], [dh]
        if jvp:
            mean, r = mean.detach(), r.detach()  # constants of the tangent, see the module's docstring
            xhat = (y32 - mean) * r
            centred = 0.0 * y32 if ty is None else ty.float() - ty.float().mean(-1, keepdim=True)
            th = r * (centred - xhat * (centred * xhat).mean(-1, keepdim=True)) * w * scale32
            outputs.append(_plus(th, _times(normed, tscale), tshift))
            cotangents.append(dth)
        g_y, g_ty, *rest = _recorded(outputs, (y, ty, scale, shift, w, b, tscale, tshift), cotangents)
        out.update(zip(("scale", "shift", "w", "b", "tscale", "tshift"), rest))
        dy, dty = _plus(dy, g_y), _plus(dty, g_ty)
    out["x"], out["tx"] = dy, dty
    if t["a"] is not None:
        out["a"] = _plus(_times(dy, t["gate"]), _times(dty, t["tgate"]))
        out["ta"] = _times(dty, t["gate"])
        rows = _plus(_times(dy, t["a"]), _times(dty, t["ta"])), _times(dty, t["a"])
        out["gate"], out["tgate"] = (None if z is None else z.float().sum(1, keepdim=True).to(z.dtype) for z in rows)
    return out


class GatedNormFunction(torch.autograd.Function):
    """``y = a gate + x`` and ``h = norm(y) (1 + scale) + shift`` with their tangents ``ty, th``.  Without ``a`` the
    norm reads ``x`` and ``y`` is None; without ``w`` there is no ``h``."""

    @staticmethod
    def forward(ctx, eps, jvp, x, a, gate, scale, shift, w, b, tx, ta, tgate, tscale, tshift):
        ctx.set_materialize_grads(False)
        ctx.eps, ctx.jvp = eps, jvp
        given = dict(x=x, a=a, tx=tx, ta=ta, w=w, b=b, gate=gate, tgate=tgate, scale=scale, tscale=tscale, shift=shift,
                     tshift=tshift)
        names = _laid_out(given)
        # (copies made here are not part of the graph that a recorded backward continues)
        ctx.as_given = all(names[n] is t for n, t in given.items())

        y, ty = _outputs(x, a is not None, a is not None and jvp)
        h, th = _outputs(x, w is not None, w is not None and jvp)
        _launch("sjvp_adaln_fwd", jvp, x.shape, eps, dict(names, y=y, ty=ty, h=h, th=th))
        if a is not None:  # the reverse mode reads y in the place of x, and without a norm neither
            given["x"] = given["tx"] = None
        ctx.names = list(given) + ["y", "ty"]
        ctx.save_for_backward(*given.values(), *((None, None) if w is None else (y, ty)))
        return y, h, ty, th

    @staticmethod
    def backward(ctx, dy, dh, dty, dth):
        if dy is None and dh is None and dty is None and dth is None:
            return (None,) * 14
        t = dict(zip(ctx.names, ctx.saved_tensors))
        if torch.is_grad_enabled():
            out = _gated_norm_recorded(t, ctx.jvp, ctx.eps, dy, dh, dty, dth)
            return (None, None, *(out.get(n) if need else None for n, need in zip(_ARGUMENTS, ctx.needs_input_grad[2:])))
        if not ctx.as_given:
            t.update(_laid_out({n: z for n, z in t.items() if n not in ("y", "ty")}))
        if t["x"] is None:
            t["x"] = t["a"]  # not read, but the call names its shape, dtype and device by x
        x, jvp = t["x"], ctx.jvp
        B, S, W = x.shape
        need = dict(zip(_ARGUMENTS, ctx.needs_input_grad[2:]))
        out = {}
        for n in ("x", "a"):
            out["d" + n], out["dt" + n] = _pair(x, need[n], need["t" + n])
        for n in _MOD:
            out["d" + n] = x.new_empty((B, 1, W)) if need[n] else None
        for n in ("w", "b"):
            out["d" + n] = torch.empty(W, device=x.device, dtype=torch.float32) if need[n] else None
        _launch("sjvp_adaln_bwd", jvp, x.shape, ctx.eps,
                dict(t, dy=_aligned(dy), dh=_aligned(dh), dty=_aligned(dty), dth=_aligned(dth), **out))
        return (None, None, *(out.get("d" + n) for n in need))


class GeluFunction(torch.autograd.Function):
    """tanh GELU and its tangent as one launch, and the reverse mode of both as one launch."""

    @staticmethod
    def forward(ctx, u, tu):
        ctx.set_materialize_grads(False)
        ctx.save_for_backward(u, tu)
        u, tu = _aligned(u), _aligned(tu)
        y, ty = _outputs(u, True, tu is not None)
        _gelu(u, tu, None, None, y, ty, 0)
        return y, ty

    @staticmethod
    def backward(ctx, dy, dty):
        if dy is None and dty is None:
            return None, None
        u, tu = ctx.saved_tensors
        if torch.is_grad_enabled():
            x, k, c = u.float(), math.sqrt(2.0 / math.pi), 0.044715
            T = torch.tanh(k * (x + c * x ** 3))
            y = 0.5 * x * (1.0 + T)
            slope = 0.5 * (1.0 + T) + 0.5 * x * (1.0 - T * T) * k * (1.0 + 3.0 * c * x * x)
            outputs = (y,) if tu is None else (y, slope * tu.float())
            return tuple(_recorded(outputs, (u, tu), (dy, dty)))
        u, tu = _aligned(u), _aligned(tu)
        du, dtu = _pair(u, True, tu is not None and dty is not None)
        _gelu(u, tu, _aligned(dy), _aligned(dty), du, dtu, 1)
        return du, dtu


class ChunkFunction(torch.autograd.Function):
    """``n`` equal pieces of the last axis of ``[B,nW]`` as ``[B,1,W]`` views; their gradients come back as one
    concatenation, where slices would each fill, copy and add a tensor of the whole size."""

    @staticmethod
    def forward(ctx, n, x):
        ctx.set_materialize_grads(False)
        ctx.shape = x.shape
        return tuple(x.detach()[:, None].chunk(n, dim=2))

    @staticmethod
    def backward(ctx, *grads):
        some = next((g for g in grads if g is not None), None)
        if some is None:
            return None, None
        return None, torch.cat([torch.zeros_like(some) if g is None else g for g in grads], dim=2).view(ctx.shape)


class PackedAttentionFunction(torch.autograd.Function):
    """Attention with the rotary embedding folded in on one ``[B,S,3,H,D]`` projection and its tangent.  The backward
    writes its gradients into one tensor of the projection's layout: three slices of it would each fill, copy
    and add a tensor of the whole size."""

    @staticmethod
    def forward(ctx, qkv, t_qkv, cos, sin):
        ctx.set_materialize_grads(False)
        B, S, _, H, D = qkv.shape
        out = _outputs(qkv, True, t_qkv is not None, (B, S, H, D))
        o, to = (None if t is None else t.transpose(1, 2) for t in out)
        q, k, v = _heads(qkv)
        mu = None
        if t_qkv is None:
            _, lse = kernels.attention_forward(q, k, v, o=o, rope=(cos, sin))
        else:
            _, _, lse, mu, _ = kernels.attention_jvp_forward(q, k, v, *_heads(t_qkv), o=o, to=to, with_li=False,
                                                             rope=(cos, sin))
        ctx.save_for_backward(qkv, t_qkv, cos, sin, *out, lse, mu)
        return out

    @staticmethod
    def backward(ctx, d_y, d_ty):
        if d_y is None and d_ty is None:
            return (None,) * 4
        run = PackedAttentionBackwardFunction.apply if torch.is_grad_enabled() else _packed_attention_backward
        return *run(d_y, d_ty, *ctx.saved_tensors), None, None


def _packed_attention_backward(d_y, d_ty, qkv, t_qkv, cos, sin, y, ty, lse, mu):
    """Gradients for the cotangents of both outputs in one launch (either may be None)."""
    d_qkv, d_t_qkv = _pair(qkv, True, d_ty is not None)
    o, to, d_o, d_to = (None if t is None else t.transpose(1, 2) for t in (y, ty, d_y, d_ty))
    tangents = (None,) * 3 if d_ty is None else _heads(t_qkv)
    if d_ty is None:
        to = mu = None
    kernels.attention_jvp_backward(*_heads(qkv), *tangents, o, to, lse, mu, dO=d_o, dTO=d_to, rope=(cos, sin),
                                   grads=(*_heads(d_qkv), *((None,) * 3 if d_ty is None else _heads(d_t_qkv))))
    return d_qkv, d_t_qkv


class PackedAttentionBackwardFunction(torch.autograd.Function):
    """The same where a graph of the backward is asked for."""

    @staticmethod
    def forward(ctx, *args):
        return _packed_attention_backward(*args)

    @staticmethod
    def backward(ctx, *grads):
        raise NotImplementedError("double backward of the attention-JVP op is not implemented")


class _CastOf(torch.autograd.Function):
    """``w16``, the values that were cast from ``w``, as part of the graph of ``w``."""

    @staticmethod
    def forward(ctx, w, w16):
        ctx.dtype = w.dtype
        return w16.view_as(w16)

    @staticmethod
    def backward(ctx, g):
        return g.to(ctx.dtype), None


class LinearFunction(torch.autograd.Function):
    """``x w^T + b`` and ``tx w^T``; in reverse mode one product for both inputs and one, summed over both in fp32, for the
    weight.  Through the general dispatch forward mode adds products with the absent tangents of weight and bias,
    zero fills and sums: 9 products per layer and step instead of 4.
    bf16 products on bf16 copies of the fp32 parameters, as autocast makes them; ``w16`` and ``b16`` are copies that are
    there already, values without a graph of their own."""

    @staticmethod
    def forward(ctx, x, tx, w, b, w16=None, b16=None):
        ctx.set_materialize_grads(False)
        w16 = w.to(x.dtype) if w16 is None else w16
        # two products, so that each output has its own storage (see _outputs); the bias enters the product's
        # accumulator: added behind it, y would be rounded twice
        y, ty = _outputs(x, shape=(*x.shape[:-1], w.shape[0]))
        rows, t_rows = x.reshape(-1, w.shape[1]), tx.reshape(-1, w.shape[1])
        if b is None:
            torch.mm(rows, w16.t(), out=y.view(-1, w.shape[0]))
        else:
            torch.addmm(b.to(x.dtype) if b16 is None else b16, rows, w16.t(), out=y.view(-1, w.shape[0]))
        torch.mm(t_rows, w16.t(), out=ty.view(-1, w.shape[0]))
        ctx.save_for_backward(x, tx, w16)
        ctx.w_dtype = w.dtype
        ctx.weight = w  # for its place in the graph; its values may have changed since
        return y, ty

    @staticmethod
    def backward(ctx, dy, dty):
        x, tx, w16 = ctx.saved_tensors
        if dy is None and dty is None:
            return (None,) * 6
        recorded = torch.is_grad_enabled()
        if recorded:
            w16 = _CastOf.apply(ctx.weight, w16)
        dx = dtx = dw = db = None
        need_x, need_tx, need_w, need_b = ctx.needs_input_grad[:4]
        if dy is not None and dty is not None:
            g, rows = _stacked(dy, dty), lambda: _stacked(x, tx)
        else:
            g = (dy if dty is None else dty).reshape(-1, w16.shape[0])
            rows = lambda: (x if dty is None else tx).reshape(-1, w16.shape[1])
        if need_x or need_tx:
            pieces = iter(torch.mm(g, w16).view(-1, *x.shape).unbind(0))
            dx = None if dy is None else next(pieces)
            dtx = None if dty is None else next(pieces)
        if need_w:
            dw = torch.mm(g.t(), rows())
        if need_b and dy is not None:
            db = dy.reshape(-1, w16.shape[0]).sum(0)
        if recorded:
            dw, db = (None if d is None else d.to(ctx.w_dtype) for d in (dw, db))
        else:
            dw, db = functional._cast_all((dw, db), (ctx.w_dtype,) * 2)
        return dx, dtx, dw, db, None, None


def _heads(qkv: Tensor):
    """The three ``[B,H,S,D]`` views of ``[B,S,3,H,D]``."""
    return qkv.permute(2, 0, 3, 1, 4).unbind(0)


@torch._dynamo.disable
def _gelu(u, tu, dy, dty, y, ty, reverse) -> None:
    host = _lib.host()
    status = host.gelu(u, tu, dy, dty, y, ty, reverse) if host else None
    if status is not None:
        return _lib.check(status)
    with torch.cuda.device(u.device):
        _lib.check(_lib.load().sjvp_gelu(*(None if t is None else t.data_ptr() for t in (u, tu, dy, dty, y, ty)), u.numel(),
                                         reverse, torch.cuda.current_stream().cuda_stream))


@torch._dynamo.disable
def bare(*modules: nn.Module) -> bool:
    """Whether calling the modules does nothing beyond the ``forward`` of their classes: no hooks of any kind, no
    ``forward`` of the instance's own, no compiled call."""
    return not _module._has_any_global_hook() and not any(
        m._forward_hooks or m._forward_pre_hooks or m._backward_hooks or m._backward_pre_hooks
        or "forward" in m.__dict__ or m._compiled_call_impl is not None for m in modules)


@torch._dynamo.disable
def serves_block(x: Tensor) -> bool:
    """Whether a block's activations are of the kind that the functions serve; cheap, asked once per block."""
    return (x.is_cuda and x.dtype == torch.bfloat16 and x.ndim == 3 and x.shape[-1] % 8 == 0
            and 8 <= x.shape[-1] <= 1024 and 0 < x.shape[0] <= 65535 and x.numel() > 0
            and torch.is_autocast_enabled("cuda") and torch.get_autocast_dtype("cuda") == torch.bfloat16
            and not torch.jit.is_tracing() and not torch.jit.is_scripting()
            and torch._C._len_torch_dispatch_stack() == 0 and torch._C._len_torch_function_stack() == 0)


def _unwrap(tensors):
    """``(interpreter or None, primals, tangents)`` on the level where both can be computed, or None where the general
    dispatch has to see the operations.  Absent tensors stay None."""
    present = [t for t in tensors if t is not None]
    if _functorch.get_interpreter_stack() is None:
        if fwAD._current_level >= 0 or any(type(t) not in (Tensor, nn.Parameter) for t in present):
            return None
        return None, list(tensors), [None] * len(tensors)
    below = _below_jvp(present)
    if below is None:
        return None
    interpreter, duals = below
    duals = iter(duals)
    pairs = [(None, None) if t is None else next(duals) for t in tensors]
    return interpreter, [p for p, _ in pairs], [t for _, t in pairs]


@torch._dynamo.disable
def gated_norm(x: Tensor, a: Optional[Tensor], gate: Optional[Tensor], norm: Optional[nn.LayerNorm],
               scale: Optional[Tensor], shift: Optional[Tensor]):
    """``(y, h)`` of :class:`GatedNormFunction` on dual or plain tensors, or None where it does not serve the call.
    The caller has asked :func:`serves_block`."""
    w = b = None
    if norm is not None:
        w, b = norm.weight, norm.bias
        if type(norm) is not nn.LayerNorm or norm.normalized_shape != x.shape[-1:] or w is None or b is None:
            return None
    found = _unwrap((x, a, gate, scale, shift, w, b))
    if found is None:
        return None
    interpreter, primals, tangents = found
    if tangents[5] is not None or tangents[6] is not None:
        return None
    B, S, W = x.shape
    for i, (p, t) in enumerate(zip(primals, tangents)):
        if p is None:
            continue
        shape, dtype = ((W,), torch.float32) if i > 4 else ((B, S, W) if i < 2 else (B, 1, W), torch.bfloat16)
        if any(z.shape != shape or z.dtype != dtype or z.device != primals[0].device for z in (p, t) if z is not None):
            return None
    eps = 0.0 if norm is None else norm.eps
    if interpreter is None:
        return GatedNormFunction.apply(eps, False, *primals, *tangents[:5])[:2]
    with interpreter.lower():
        y, h, ty, th = GatedNormFunction.apply(eps, True, *primals, *tangents[:5])
    return tuple(None if p is None else _dual_above(interpreter, p, t) for p, t in ((y, ty), (h, th)))


@torch._dynamo.disable
def gelu(u: Tensor) -> Optional[Tensor]:
    """tanh GELU of a dual or plain bf16 tensor, or None where it is not served.  The caller has asked
    :func:`serves_block` on the block's input."""
    if u.dtype != torch.bfloat16 or u.numel() % 8 or not u.is_cuda:
        return None
    found = _unwrap((u,))
    if found is None:
        return None
    interpreter, (p,), (t,) = found
    if interpreter is None:
        return GeluFunction.apply(p, None)[0]
    if t.dtype != p.dtype or t.shape != p.shape:
        return None
    with interpreter.lower():
        y, ty = GeluFunction.apply(p, t)
    return _dual_above(interpreter, y, ty)


@torch._dynamo.disable
def cast(*layers: nn.Linear):
    """``{layer: (weight, bias)}`` with bf16 copies of the fp32 parameters of linear layers for :func:`linear` and
    :func:`plain_linear`, made by one launch where autocast would cast one by one (and once more for each use under forward
    mode), or None where that is not served.  The caller has asked :func:`serves_block`.

    Under forward mode the copies are values without a graph, :func:`linear` takes the parameters beside them; in a plain call that
    records gradients each has a node of its own.  (One node for all would compute the gradients of frozen parameters too, and
    hand over none before the last is there.)  Both are made anew for each call.  A plain call that records none takes what
    autocast keeps for its region, the casts of leaves that require a gradient, from there: None where that is all, else such
    parameters stand for themselves in the result.  Network without
    gradients, ms a call in a region of ten calls (of one), casts of its own / the region's: text8 32 samples 5.34 (5.53) / 5.13
    (6.12), 128 8.95 (9.36) / 8.87 (9.55); LM1B 32 samples 4.24 (4.51) / 4.04 (5.01), 128 7.35 (7.64) / 7.33 (7.86)."""
    stack = _functorch.get_interpreter_stack()
    if stack is None:
        if fwAD._current_level >= 0:
            return None
    elif len(stack) != 1 or stack[0].key() != functional.TransformType.Jvp:
        return None
    if not all(type(m) is nn.Linear for m in layers):
        return None
    params = [p for m in layers for p in (m.weight, m.bias) if p is not None]
    own = params
    if stack is None and not torch.is_grad_enabled() and torch.is_autocast_enabled("cuda") and torch.is_autocast_cache_enabled():
        own = [None if p.requires_grad and p.is_leaf else p for p in params]
        if all(p is None for p in own):
            return None
    if not bare(*layers):
        return None
    if any(type(p) not in (Tensor, nn.Parameter) or p.dtype != torch.float32 or p.device != params[0].device or not p.is_cuda
           or _functorch.is_functorch_wrapped_tensor(p) for p in params):
        return None
    if stack is None and torch.is_grad_enabled() and any(p.requires_grad for p in params):
        copies = _lib.host().cast(params, torch.bfloat16, True) if _lib.host() else None
        if copies is None:
            return None
        copies = iter(kernels._host_result(copies))
    else:
        below = contextlib.nullcontext() if stack is None else functional.retrieve_current_functorch_interpreter().lower()
        with below, torch.no_grad():
            made = functional._cast_all(own, (torch.bfloat16,) * len(params))
        copies = iter([p if c is None else c for p, c in zip(params, made)])
    return {m: (next(copies), None if m.bias is None else next(copies)) for m in layers}


@torch._dynamo.disable
def linear(layer: nn.Linear, x: Tensor, copies=None) -> Optional[Tensor]:
    """The layer on a dual tensor, with the ``copies`` of :func:`cast` where there are any, or None where it is not served (a
    plain tensor included: that is one product already).  The caller has asked :func:`serves_block`."""
    if x.dtype != torch.bfloat16 or _functorch.get_interpreter_stack() is None:
        return None
    if copies is None and (type(layer) is not nn.Linear or not bare(layer)):
        return None
    w, b = layer.weight, layer.bias
    found = _unwrap((x, w, b))
    if found is None:
        return None
    interpreter, (p, w, b), (t, *absent) = found
    if t is None or any(z is not None for z in absent) or t.dtype != p.dtype or t.shape != p.shape or p.numel() == 0 \
            or any(z.dtype != torch.float32 or z.device != p.device for z in (w, b) if z is not None):
        return None
    with interpreter.lower():
        y, ty = LinearFunction.apply(p, t, w, b, *(() if copies is None else copies[layer]))
    return _dual_above(interpreter, y, ty)


@torch._dynamo.disable
def plain_linear(layer: nn.Linear, x: Tensor, copies) -> Optional[Tensor]:
    """The layer on a plain tensor with the copies of :func:`cast`; None inside a transform."""
    return None if _functorch.get_interpreter_stack() is not None else nn.functional.linear(x, *copies[layer])


@torch._dynamo.disable
def chunk(x: Tensor, n: int):
    """``x[:, None].chunk(n, dim=2)`` of a dual or plain ``[B,nW]`` tensor, or None where it is not served.  The caller has
    asked :func:`serves_block`."""
    found = _unwrap((x,)) if x.ndim == 2 and x.shape[1] % n == 0 and x.dtype == torch.bfloat16 else None
    if found is None:
        return None
    interpreter, (p,), (t,) = found
    if interpreter is None:
        return ChunkFunction.apply(n, p)
    with interpreter.lower():
        primals, tangents = ChunkFunction.apply(n, p), ChunkFunction.apply(n, t)
    return tuple(_dual_above(interpreter, a, b) for a, b in zip(primals, tangents))


@torch._dynamo.disable
def attention(qkv: Tensor, cos: Tensor, sin: Tensor) -> Optional[Tensor]:
    """``safe_sdpa_jvp_rotary`` of the three slices of a dual or plain ``[B,S,3,H,D]`` projection, ``[B,S,H,D]``, or
    None where it is not served.  The caller has asked :func:`serves_block`."""
    # tables sliced inside the transform are wrapped like everything computed there
    found = _unwrap((qkv, cos, sin)) if functional.AUTOGRAD_WIRING != "reference" else None
    if found is None:
        return None
    interpreter, (p, cos, sin), (t, *tables) = found
    if any(z is not None for z in tables) or (t is None) != (interpreter is None):
        return None
    if p.dtype != torch.bfloat16 or any(z.ndim != 5 or z.shape != p.shape or z.dtype != p.dtype or not z.is_contiguous()
                                        for z in (p, t) if z is not None) or cos.requires_grad or sin.requires_grad:
        return None
    if interpreter is None:
        q, k, v = _heads(p.detach())
        return PackedAttentionFunction.apply(p, None, cos, sin)[0] \
            if kernels.rotary_fusable(q, k, cos, (v,), sin=sin) else None
    with interpreter.lower():
        q, k, v = _heads(p.detach())
        if not kernels.rotary_fusable(q, k, cos, (v, *_heads(t.detach())), sin=sin):
            return None
        y, ty = PackedAttentionFunction.apply(p, t, cos, sin)
    return _dual_above(interpreter, y, ty)
