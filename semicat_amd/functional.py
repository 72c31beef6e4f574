"""Autograd surface of the attention-JVP op: ``sdpa_jvp`` / ``safe_sdpa_jvp`` with the semantics of
olsdavis/semicat's ``semicat/jvp_utils/functional.py`` (cited by line below), backed by the HIP
kernels in :mod:`semicat_amd.kernels`.

How the op is wired (same shape as the reference, functional.py:216-307):

* ``SDPAFunction.forward`` only allocates the primal output ``y`` and the statistic ``M``
  (functional.py:218-231); under forward-mode AD its ``jvp`` runs the fused kernel once, which
  fills ``y`` and ``M`` in place and returns the tangent ``t_y`` (functional.py:240-258).
* ``SDPAJVPForwardFunction`` is the reverse-mode node of the tangent output: its backward receives
  the cotangent on ``t_y`` and returns gradients for q, k, v and the three tangents
  (functional.py:52-87).
* ``SDPAFunction.backward`` is the reverse-mode node of the primal output (functional.py:261-268).

Beyond the reference: called without forward-mode tangents the reference returns an uninitialised
``y`` (functional.py:286-287); here that case is detected and a primal-only kernel computes ``y``
(and supports reverse mode), so the op is a strict superset.  A missing tangent is treated as zero.

Two wirings of the same op exist; ``AUTOGRAD_WIRING`` selects the one ``sdpa_jvp`` uses:

* ``"fused"`` (default): the dual inputs are unpacked, ONE autograd node (``SDPAFusedFunction``)
  produces ``y`` and ``t_y`` with one forward launch, and the two are handed back as a dual tensor.
  Reverse mode then reaches that node once, with the cotangents of both outputs, and runs the
  backward as ONE launch (the six gradients are accumulated in fp32 and rounded once).
* ``"reference"``: the reference's three-function arrangement as described above, in which the node
  of ``y`` and the node of ``t_y`` each launch the backward with their own cotangent and autograd
  adds the two 16-bit results for q, k, v.
"""
from __future__ import annotations

from typing import Any, Optional

import torch
import torch.autograd.forward_ad as fwAD
from torch import Tensor
from torch._C import _functorch
from torch._functorch.pyfunctorch import TransformType, retrieve_current_functorch_interpreter

from . import _lib, kernels


AUTOGRAD_WIRING = "fused"  # or "reference"
# How safe_sdpa_jvp serves float32 callers with bf16 arithmetic (functional.py:318-332):
#   "torch"   (default) casts around the 16-bit kernels, as the reference does; under one torch.func.jvp all tensors of a
#             direction are cast by one launch (csrc/sjvp_cast.hip), with the bits that torch casts give;
#   "library" the library's multi-tensor cast launches around them (half the launches, no kernel that is
#             not the library's own);
#   "folded"  the float32 tensors handed to the kernels, which round as they load and store float32 (SJVP_FP32_BF16).
# "folded" is not the default: autograd keeps the caller's own tensors for it, so they (and the result) may not be
# written to before the backward, they stay in memory at twice the size (B=64 H=12 L=128 D=64: 191 MB held by a call on
# temporaries against 145), the last dimension has to have unit stride, and it is the faster route for short sequences
# at D = 64 only.  Measured on an MI355X, forward + backward under torch.func.jvp in microseconds, folded / casts:
#   D = 64:  B=64 H=12 L=128 187 / 280, B=8 H=16 L=1024 604 / 621, L=2048 2125 / 2010, L=4096 7936 / 7410;
#   D = 128: B=8 H=16 L=1024 1508 / 1260, L=2048 5496 / 4136, L=4096 20085 / 14900.
FP32_CALLERS = "torch"


def _has_tangent(t: Tensor) -> bool:
    return fwAD.unpack_dual(t).tangent is not None


class SDPAJVPFlashBackwardFunction(torch.autograd.Function):
    """Gradients for the cotangent on the tangent output (functional.py:90-168)."""

    @staticmethod
    def forward(ctx, q, k, v, t_q, t_k, t_v, tangents_t_o, lse, mu, o, t_o):
        dq, dk, dv, dtq, dtk, dtv = kernels.attention_jvp_backward(
            q, k, v, t_q, t_k, t_v, o, t_o, lse, mu, dO=None, dTO=tangents_t_o)
        return dq, dk, dv, dtq, dtk, dtv

    @staticmethod
    def backward(ctx, *grads):
        raise NotImplementedError("double backward of the attention-JVP op is not implemented")


class SDPABackwardFunction(torch.autograd.Function):
    """Gradients for the cotangent on the primal output (functional.py:171-213)."""

    @staticmethod
    def forward(ctx, q, k, v, o, do, M, arith=None, cos=None, sin=None):
        dq, dk, dv, _, _, _ = kernels.attention_jvp_backward(
            q, k, v, None, None, None, o, None, M, None, dO=do, dTO=None, arithmetic=arith,
            rope=None if cos is None else (cos, sin))
        return dq, dk, dv

    @staticmethod
    def backward(ctx, *grads):
        raise NotImplementedError("double backward of the attention-JVP op is not implemented")


class SDPAJVPForwardFunction(torch.autograd.Function):
    """Runs the fused forward; node of the tangent output (functional.py:52-87)."""

    @staticmethod
    def forward(q, k, v, t_q, t_k, t_v, y, M):
        # y and M (allocated by SDPAFunction.forward) are filled in place by the fused kernel.
        # LI, which the reference also keeps (functional.py:57-59), is not needed by the backward.
        with torch.no_grad():
            # the tangent output takes the memory layout of the primal output
            _, t_y, _, MU, _ = kernels.attention_jvp_forward(q, k, v, t_q, t_k, t_v, o=y,
                                                             to=torch.empty_like(y), lse=M, with_li=False)
        return t_y, MU

    @staticmethod
    def setup_context(ctx, inputs: tuple[Any, ...], output: Any) -> Any:
        t_y, MU = output
        ctx.save_for_backward(*inputs, t_y, MU)
        ctx.mark_non_differentiable(MU)

    @staticmethod
    def backward(ctx, d_t_y, *args):
        q, k, v, t_q, t_k, t_v, y, M, t_y, MU = ctx.saved_tensors
        if d_t_y is None:
            return (None,) * 8
        grads = SDPAJVPFlashBackwardFunction.apply(q, k, v, t_q, t_k, t_v, d_t_y, M, MU, y, t_y)
        return *grads, None, None


def _empty_output(q: Tensor, d_v: int, seq_major: bool) -> Tensor:
    """A ``[B,H,S,D]`` output buffer: contiguous as the reference allocates it (functional.py:224-227),
    or, for callers that work in ``[B,S,H,D]``, a view of a ``[B,S,H,D]``-contiguous buffer, so that
    handing the result back in their layout needs no copy (the kernels write through strides)."""
    B, H, S, _ = q.shape
    if seq_major:
        return torch.empty((B, S, H, d_v), device=q.device, dtype=q.dtype).transpose(1, 2)
    return torch.empty((B, H, S, d_v), device=q.device, dtype=q.dtype)


class SDPAFunction(torch.autograd.Function):
    """The op under forward-mode AD (functional.py:216-268)."""

    @staticmethod
    def forward(q, k, v, seq_major=False):
        y = _empty_output(q, v.shape[-1], seq_major)
        M = torch.empty((q.shape[0], q.shape[1], kernels.stat_rows(q.shape[2])), device=q.device,
                        dtype=torch.float32)
        return y, M

    @staticmethod
    def setup_context(ctx: Any, inputs: tuple[Any, ...], output: Any) -> Any:
        ctx.save_for_forward(*inputs[:3], *output)
        ctx.save_for_backward(*inputs[:3], *output)
        ctx.set_materialize_grads(False)

    @staticmethod
    def jvp(ctx, t_q, t_k, t_v, *_):
        q, k, v, y, M = ctx.saved_for_forward
        t_q = torch.zeros_like(q) if t_q is None else t_q
        t_k = torch.zeros_like(k) if t_k is None else t_k
        t_v = torch.zeros_like(v) if t_v is None else t_v
        t_y, _ = SDPAJVPForwardFunction.apply(q, k, v, t_q, t_k, t_v, y, M)
        return t_y, torch.zeros_like(M)

    @staticmethod
    def backward(ctx, d_y, d_M):
        if d_y is None:
            return None, None, None, None
        q, k, v, y, M = ctx.saved_tensors
        with torch.no_grad():
            dq, dk, dv = SDPABackwardFunction.apply(q, k, v, y, d_y, M)
        return dq, dk, dv, None


class SDPAFusedFunction(torch.autograd.Function):
    """``(q, k, v, t_q, t_k, t_v) -> (y, t_y)`` as one autograd node: one fused forward launch, and
    in reverse mode one backward launch that takes the cotangents of both outputs (either may be
    absent).  Replaces the pair functional.py:52-87 / 216-268 when the caller's dual tensors are
    unpacked by hand (see ``_sdpa``)."""

    @staticmethod
    def forward(q, k, v, t_q, t_k, t_v, seq_major=False, arith=None, cos=None, sin=None):
        y = _empty_output(q, v.shape[-1], seq_major)
        y, t_y, M, MU, _ = kernels.attention_jvp_forward(q, k, v, t_q, t_k, t_v, o=y, to=torch.empty_like(y),
                                                         with_li=False, arithmetic=arith,
                                                         rope=None if cos is None else (cos, sin))
        return y, t_y, M, MU

    @staticmethod
    def setup_context(ctx: Any, inputs: tuple[Any, ...], output: Any) -> Any:
        y, t_y, M, MU = output
        ctx.rope = inputs[8] is not None
        ctx.save_for_backward(*inputs[:6], y, t_y, M, MU, *(inputs[8:10] if ctx.rope else ()))
        ctx.arith = inputs[7]
        ctx.mark_non_differentiable(M, MU)
        ctx.set_materialize_grads(False)

    @staticmethod
    def backward(ctx, d_y, d_t_y, *_):
        if d_y is None and d_t_y is None:
            return (None,) * 10
        q, k, v, t_q, t_k, t_v, y, t_y, M, MU, *rope = ctx.saved_tensors
        cos, sin = rope if ctx.rope else (None, None)
        with torch.no_grad():
            if d_t_y is None:
                dq, dk, dv = SDPABackwardFunction.apply(q, k, v, y, d_y, M, ctx.arith, cos, sin)
                return dq, dk, dv, None, None, None, None, None, None, None
            grads = SDPAJVPFusedBackwardFunction.apply(q, k, v, t_q, t_k, t_v, y, t_y, M, MU, d_y, d_t_y,
                                                       ctx.arith, cos, sin)
        return *grads, None, None, None, None


class SDPAJVPFusedBackwardFunction(torch.autograd.Function):
    """Gradients for cotangents on both outputs in one launch (``d_y`` may be None)."""

    @staticmethod
    def forward(ctx, q, k, v, t_q, t_k, t_v, y, t_y, M, MU, d_y, d_t_y, arith=None, cos=None, sin=None):
        return kernels.attention_jvp_backward(q, k, v, t_q, t_k, t_v, y, t_y, M, MU, dO=d_y, dTO=d_t_y,
                                              arithmetic=arith, rope=None if cos is None else (cos, sin))

    @staticmethod
    def backward(ctx, *grads):
        raise NotImplementedError("double backward of the attention-JVP op is not implemented")


class SDPAPrimalFunction(torch.autograd.Function):
    """The op without forward-mode tangents: plain attention with the primal-only kernels."""

    @staticmethod
    def forward(ctx, q, k, v, seq_major=False, arith=None, cos=None, sin=None):
        rope = None if cos is None else (cos, sin)
        y, M = kernels.attention_forward(q, k, v, o=_empty_output(q, v.shape[-1], seq_major), arithmetic=arith,
                                         rope=rope)
        ctx.save_for_backward(q, k, v, y, M, *(rope or ()))
        ctx.arith = arith
        return y

    @staticmethod
    def backward(ctx, d_y):
        q, k, v, y, M, *rope = ctx.saved_tensors
        dq, dk, dv = SDPABackwardFunction.apply(q, k, v, y, d_y, M, ctx.arith, *rope)
        return dq, dk, dv, None, None, None, None


def _cast_all(tensors, dtypes):
    """``[t.to(dtype)]`` of present tensors, for a caller that records nothing: through the library's multi-tensor cast (one
    launch, 6 us of host time for six tensors) where it serves them, else with one multi-tensor copy (22 us)."""
    tensors = list(tensors)
    if len(set(dtypes)) == 1 and any(t is not None and t.is_cuda for t in tensors) and _lib.host():
        native = kernels._host_result(_lib.host().cast(tensors, dtypes[0]))
        if native is not None:
            return native
    out = [t if t is None or t.dtype == dtype else torch.empty_like(t, dtype=dtype) for t, dtype in zip(tensors, dtypes)]
    pairs = [(o, t) for o, t in zip(out, tensors) if o is not t]
    if pairs:
        torch._foreach_copy_(*map(list, zip(*pairs)))
    return out


class SDPASeqMajorFunction(torch.autograd.Function):
    """:class:`SDPAFusedFunction` on ``[B,S,H,D]`` tensors, for tensors below the forward-mode level (see
    :func:`_below_jvp`): the change of axes, and the casts to the dtype ``compute`` and back, happen in here, where they
    leave no autograd nodes.  With ``compute`` only its copies are kept for the backward: the caller may write to its
    own tensors and to the result.  With ``apart`` the rotation by ``cos``, ``sin`` is a launch of its own in front of the
    attention kernels (and behind them in reverse mode) instead of folded into them; the rotated tensors are what is kept."""

    @staticmethod
    def forward(ctx, q, k, v, t_q, t_k, t_v, arith, cos, sin, compute, apart=False):
        ctx.rope = None if cos is None or apart else (cos, sin)
        ctx.arith, ctx.compute, ctx.apart = arith, compute, apart
        given = (q, k, v, t_q, t_k, t_v)
        ctx.dtypes = [t.dtype for t in given]
        if compute is not None:
            given = _cast_all(given, (compute,) * 6)
        if apart:
            q, k, t_q, t_k = kernels.rotary_embedding((q, k, t_q, t_k), cos, sin)
            given = (q, k, v, t_q, t_k, t_v)
        B, S, H, _ = q.shape
        y, t_y = (torch.empty((B, S, H, v.shape[-1]), device=q.device, dtype=given[0].dtype) for _ in range(2))
        *inputs, o, to = (t.transpose(1, 2) for t in (*given, y, t_y))
        _, _, M, MU, _ = kernels.attention_jvp_forward(*inputs, o=o, to=to, with_li=False, arithmetic=arith,
                                                       rope=ctx.rope)
        ctx.save_for_backward(*given, y, t_y, M, MU, *(() if cos is None else (cos, sin)))
        ctx.rope = ctx.rope is not None
        ctx.set_materialize_grads(False)
        return (y, t_y) if compute is None else tuple(_cast_all((y, t_y), (q.dtype,) * 2))

    @staticmethod
    def backward(ctx, d_y, d_t_y):
        if d_y is None and d_t_y is None:
            return (None,) * 11
        *tensors, M, MU = ctx.saved_tensors[:10]
        tables = ctx.saved_tensors[10:]
        rope = tables if ctx.rope else None
        with torch.no_grad():
            q, k, v, t_q, t_k, t_v, y, t_y = (t.transpose(1, 2) for t in tensors)
            if ctx.compute is not None:
                d_y, d_t_y = _cast_all((d_y, d_t_y), (ctx.compute,) * 2)
            d_y, d_t_y = (None if d is None else d.transpose(1, 2) for d in (d_y, d_t_y))
            grads = kernels.attention_jvp_backward(q, k, v, t_q, t_k, t_v, y, t_y, M, MU, dO=d_y, dTO=d_t_y,
                                                   arithmetic=ctx.arith, rope=rope)
            grads = [None if g is None else g.transpose(1, 2) for g in grads]
            if ctx.apart:
                turned = [i for i in (0, 1, 3, 4) if grads[i] is not None]
                for i, g in zip(turned, kernels.rotary_embedding([grads[i] for i in turned], *tables, inverse=True)):
                    grads[i] = g
            return *_cast_all(grads, ctx.dtypes), None, None, None, None, None


def _below_jvp(tensors):
    """``(interpreter, [(primal, tangent)])`` of tensors inside ONE ``torch.func.jvp`` and no other transform, taken
    off that level: plain tensors on which autograd records as it does outside.  None anywhere else (no transform,
    several, vmap, grad, subclasses of Tensor).

    An ``autograd.Function`` applied inside the transform goes through functorch's general dispatch, which builds a
    class per call, flattens and rewraps trees and binds signatures: 0.3 of the 0.55 ms of a forward + backward at
    B=64 H=12 L=128 D=64 on fp32 tensors, whose kernels take 0.14 ms.  The op knows its own tangents, so
    it can compute both outputs below the level and wrap them."""
    stack = _functorch.get_interpreter_stack()
    if stack is None or len(stack) != 1 or stack[0].key() != TransformType.Jvp:
        return None
    level, duals, any_tangent = stack[0].level(), [], False
    for t in tensors:
        tangent = None
        if _functorch.is_functorch_wrapped_tensor(t):
            if _functorch.maybe_get_level(t) != level:
                return None
            tangent = fwAD.unpack_dual(t).tangent
            t = _functorch.get_unwrapped(t)
            if tangent is not None:
                any_tangent = True
                if _functorch.is_functorch_wrapped_tensor(tangent):
                    tangent = _functorch.get_unwrapped(tangent)
                if type(tangent) not in (Tensor, torch.nn.Parameter) or tangent._is_zerotensor():
                    return None
        if type(t) not in (Tensor, torch.nn.Parameter) or _functorch.is_functorch_wrapped_tensor(t):
            return None
        duals.append((t, tangent))
    return (retrieve_current_functorch_interpreter(), duals) if any_tangent else None


def _dual_above(interpreter, primal: Tensor, tangent: Tensor) -> Tensor:
    """The dual tensor, on the level of the transform, of two tensors below it."""
    wrapped = (_functorch._wrap_for_grad(t, interpreter.level()) for t in (primal, tangent))
    return fwAD.make_dual(*wrapped)


@torch._dynamo.disable
def _sdpa_seq_major(q: Tensor, k: Tensor, v: Tensor, arith: Optional[str] = None, cos: Optional[Tensor] = None,
                    sin: Optional[Tensor] = None) -> Tensor:
    """The op on ``[B,S,H,D]`` tensors.  With ``cos``, ``sin`` the caller has asked ``rotary_fusable``."""
    below = _below_jvp((q, k, v)) if AUTOGRAD_WIRING != "reference" else None
    if below is None:
        return _sdpa(q.transpose(1, 2), k.transpose(1, 2), v.transpose(1, 2), seq_major=True, arith=arith, cos=cos,
                     sin=sin).transpose(1, 2)
    return _seq_major_below(below, arith, cos, sin)


def _seq_major_below(below, arith=None, cos=None, sin=None, compute=None, apart=False) -> Tensor:
    interpreter, duals = below
    with interpreter.lower():
        primals = [p for p, _ in duals]
        tangents = [torch.zeros_like(p) if t is None else t for p, t in duals]
        y, t_y = SDPASeqMajorFunction.apply(*primals, *tangents, arith, cos, sin, compute, apart)
    return _dual_above(interpreter, y, t_y)


@torch._dynamo.disable
def _sdpa_cast_below(q: Tensor, k: Tensor, v: Tensor) -> Optional[Tensor]:
    """The op in bfloat16 with its casts below the level of one ``torch.func.jvp``, or None where the casts have to be
    seen.  (As duals each of the casts and its derivative would go through the transform: forward + backward at
    B=64 H=12 L=128 D=64 690 against 370 us.)"""
    below = _below_jvp((q, k, v)) if AUTOGRAD_WIRING != "reference" else None
    return None if below is None else _seq_major_below(below, compute=torch.bfloat16)


@torch._dynamo.disable
def sdpa_jvp(q: Tensor, k: Tensor, v: Tensor) -> Tensor:
    """Fused scaled-dot-product attention with forward-mode (jvp) support; ``[B,H,S,D]`` bf16/fp16
    (functional.py:272-307).  Usage: ``y, t_y = torch.func.jvp(sdpa_jvp, (q, k, v), (t_q, t_k, t_v))``
    or wrap a whole model that calls it in ``torch.func.jvp``; both outputs support ``backward``."""
    return _sdpa(q, k, v, seq_major=False)


@torch._dynamo.disable
def _sdpa(q: Tensor, k: Tensor, v: Tensor, seq_major: bool, arith: Optional[str] = None,
          cos: Optional[Tensor] = None, sin: Optional[Tensor] = None) -> Tensor:
    if _has_tangent(q) or _has_tangent(k) or _has_tangent(v):
        if AUTOGRAD_WIRING == "reference":
            if cos is not None:
                raise ValueError("the reference wiring has no folded rotary embedding")
            y, _ = SDPAFunction.apply(q, k, v, seq_major)
            return y
        (q, t_q), (k, t_k), (v, t_v) = (fwAD.unpack_dual(t) for t in (q, k, v))
        t_q = torch.zeros_like(q) if t_q is None else t_q
        t_k = torch.zeros_like(k) if t_k is None else t_k
        t_v = torch.zeros_like(v) if t_v is None else t_v
        y, t_y, _, _ = SDPAFusedFunction.apply(q, k, v, t_q, t_k, t_v, seq_major, arith, cos, sin)
        return fwAD.make_dual(y, t_y)
    return SDPAPrimalFunction.apply(q, k, v, seq_major, arith, cos, sin)


def safe_sdpa_jvp(q: Tensor, k: Tensor, v: Tensor, precise: bool = False) -> Tensor:
    """``[B,S,H,D]`` wrapper with the reference's dtype policy (functional.py:310-332): inputs that
    are neither bf16 nor fp16 are computed in bfloat16 and the result comes back in their dtype, cast
    with torch as in the reference; for float32 inputs ``FP32_CALLERS`` selects two other routes (the
    library's own cast launches, or float32 tensors handed to the kernels as they are; figures beside
    it).  ``precise=True`` runs float32 inputs in the
    library's fp32 mode instead (contractions of fp32 accuracy, about 1e-6 against fp64; four to five
    times the time of the 16-bit kernels)."""
    orig_dtype = q.dtype
    arith = None
    fp32_bf16 = orig_dtype == torch.float32 and not precise and AUTOGRAD_WIRING != "reference" \
        and k.dtype == torch.float32 and v.dtype == torch.float32
    if fp32_bf16 and FP32_CALLERS == "library" and q.is_cuda:
        from .rotary import cast_tensors
        q, k, v = cast_tensors((q, k, v), torch.bfloat16)
        y = _sdpa(q.transpose(1, 2), k.transpose(1, 2), v.transpose(1, 2), seq_major=True).transpose(1, 2)
        return cast_tensors(y, orig_dtype)
    if fp32_bf16 and FP32_CALLERS == "folded":
        arith = "bf16"
    elif orig_dtype != torch.bfloat16 and orig_dtype != torch.float16 and not (precise and orig_dtype == torch.float32):
        y = _sdpa_cast_below(q, k, v)
        if y is not None:
            return y
        q = q.to(torch.bfloat16)
        k = k.to(torch.bfloat16)
        v = v.to(torch.bfloat16)
    # The reference returns a [B,S,H,D] view of a [B,H,S,D]-contiguous result, which its callers then
    # copy when they flatten the heads (duo.py:155); here the kernels write [B,S,H,D] memory directly.
    y = _sdpa_seq_major(q, k, v, arith)
    if y.dtype != orig_dtype:
        y = y.to(orig_dtype)
    return y


@torch._dynamo.disable
def safe_sdpa_jvp_rotary(q: Tensor, k: Tensor, v: Tensor, cos: Tensor, sin: Tensor) -> Tensor:
    """``safe_sdpa_jvp(rot(q), rot(k), v)`` for ``[B,S,H,D]`` tensors (views of a fused projection are
    fine), where ``rot`` is the rotary position embedding that semicat/net/duo.py:45-55 applies to q and
    k in front of the op, with fp32 ``cos``/``sin`` tables ``[S, D/2]``.  Where the kernels serve the
    shape (head dimension 64, at most 128 keys, bf16 / fp16 inputs with aligned rows) the rotation is
    folded into the attention launches: q and k are read unrotated, rotated on chip, and the gradients
    come back through the inverse rotation, so no rotary launch and no rotated copy of q, k exists in
    either AD mode.  Other shapes rotate with the library's rotary kernel first."""
    below = _below_jvp((q, k, v)) if AUTOGRAD_WIRING != "reference" else None
    if below is not None:
        interpreter, duals = below
        with interpreter.lower():
            (qh, tq), (kh, tk), (vh, tv) = [[None if t is None else t.transpose(1, 2) for t in d] for d in duals]
            plain = not _functorch.is_functorch_wrapped_tensor(cos) and not _functorch.is_functorch_wrapped_tensor(sin)
            fusable = plain and kernels.rotary_fusable(qh, kh, cos, (vh, tq, tk, tv), sin=sin)
        if fusable:
            return _seq_major_below(below, None, cos, sin)
        if plain and q.dtype in (torch.bfloat16, torch.float16) and all(
                z.dtype == q.dtype and z.ndim == 4 for pair in duals for z in pair if z is not None):
            # The rotary launch below the level too: as a function of its own under the transform it goes through functorch's
            # general dispatch three times (forward + backward at B=4 H=12 S=256 D=64 1160 us, here 427).
            return _seq_major_below(below, None, cos, sin, apart=True)
    qh, kh, vh = q.transpose(1, 2), k.transpose(1, 2), v.transpose(1, 2)
    tangents = [fwAD.unpack_dual(t).tangent for t in (qh, kh, vh)]
    if AUTOGRAD_WIRING != "reference" and kernels.rotary_fusable(
            fwAD.unpack_dual(qh).primal, fwAD.unpack_dual(kh).primal, cos,
            [fwAD.unpack_dual(vh).primal, *tangents], sin=sin):
        return _sdpa(qh, kh, vh, seq_major=True, cos=cos, sin=sin).transpose(1, 2)
    from .rotary import apply_rotary
    q, k = apply_rotary((q, k), cos, sin)
    return safe_sdpa_jvp(q, k, v)
