"""torch.library registration of the attention core: ``chia_attn::fwd`` and ``chia_attn::bwd``.

The reference's kernels are plain Python functions that launch on torch's
current stream (extra_bench.py:12,19); torch.compile traces into them and
breaks its graph at the launch.  Registered as custom operators with fake
(shape-only) implementations and an autograd formula, the core is one opaque
node to torch.compile, make_fx and AOTAutograd -- the "operators Inductor does
not cover" use of the reference's README.md:3-6 -- and gradients flow through
the registered backward.

  chia_attn::fwd(q, k, v, <mask and score parameters>) -> (o, lse)
      o: bf16 like q; lse: float32 [B, H, S] (natural log, softmax only; an
      empty [0] tensor for sigmoid / ReLU).  lse is not differentiable.
  chia_attn::bwd(do, q, k, v, o, lse, <parameters>) -> (dq, dk, dv)

Per-head vectors are optional float32 device tensors [H]; ``scale`` None
stands for the default 1 / sqrt(head_dim).  Both operators run
``chia_attn_fwd_lse`` / ``chia_attn_bwd`` of libchia_attn.so on torch's current
stream, and raise if the library is not built.
"""
from __future__ import annotations

from typing import Optional, Tuple

import torch
from torch import Tensor


NAMESPACE = "chia_attn"


def _params(norm, causal, window, dilation, block, prefix, scale, head_scale, alibi_slopes, softcap, bias,
            post_scale) -> dict:
    return dict(norm=norm, causal=causal, window=window, dilation=dilation, block=block, prefix=prefix,
                scale=scale, head_scale=head_scale, alibi_slopes=alibi_slopes,
                softcap=softcap, bias=bias, post_scale=post_scale)


@torch.library.custom_op(f"{NAMESPACE}::fwd", mutates_args=(), device_types="cuda")
def fwd(q: Tensor, k: Tensor, v: Tensor, norm: str, causal: bool, window: int, dilation: int, block: int,
        prefix: int, scale: Optional[float], head_scale: Optional[Tensor], alibi_slopes: Optional[Tensor],
        softcap: float, bias: float, post_scale: float) -> Tuple[Tensor, Tensor]:
    from .attention import run_forward

    return run_forward(q, k, v, _params(norm, causal, window, dilation, block, prefix, scale, head_scale,
                                        alibi_slopes, softcap, bias, post_scale))


@fwd.register_fake
def _fwd_fake(q, k, v, norm, causal, window, dilation, block, prefix, scale, head_scale, alibi_slopes, softcap,
              bias, post_scale):
    torch._check(q.dim() == 4, lambda: "q must be 4-D [B, H, S, D]")
    B, H, S, _ = q.shape
    lse_shape = (B, H, S) if norm == "softmax" else (0,)
    return torch.empty_like(q, memory_format=torch.contiguous_format), q.new_empty(lse_shape, dtype=torch.float32)


@torch.library.custom_op(f"{NAMESPACE}::bwd", mutates_args=(), device_types="cuda")
def bwd(do: Tensor, q: Tensor, k: Tensor, v: Tensor, o: Tensor, lse: Tensor, norm: str, causal: bool, window: int,
        dilation: int, block: int, prefix: int, scale: Optional[float], head_scale: Optional[Tensor],
        alibi_slopes: Optional[Tensor], softcap: float, bias: float, post_scale: float
        ) -> Tuple[Tensor, Tensor, Tensor]:
    from .attention import run_backward

    p = _params(norm, causal, window, dilation, block, prefix, scale, head_scale, alibi_slopes, softcap, bias,
                post_scale)
    return run_backward(do, q, k, v, o, lse if lse.numel() else None, p)


@bwd.register_fake
def _bwd_fake(do, q, k, v, o, lse, norm, causal, window, dilation, block, prefix, scale, head_scale, alibi_slopes,
              softcap, bias, post_scale):
    return (torch.empty_like(q, memory_format=torch.contiguous_format),
            torch.empty_like(k, memory_format=torch.contiguous_format),
            torch.empty_like(v, memory_format=torch.contiguous_format))


def _setup_context(ctx, inputs, output):
    q, k, v, *rest = inputs
    o, lse = output
    ctx.rest = rest  # norm .. post_scale, schema order (per-head tensors included)
    ctx.save_for_backward(q, k, v, o, lse)
    ctx.mark_non_differentiable(lse)
    ctx.set_materialize_grads(False)  # no zero-filled gradient for the unused lse


_DK = torch._C.DispatchKey
# The dispatch keys of a CUDA tensor whose memory holds its values.
_PLAIN_KEYS = (torch._C.DispatchKeySet(_DK.CUDA).add(_DK.ADInplaceOrView).add(_DK.AutogradCUDA)
               .add(_DK.AutocastCUDA))


def _holds_values(t: Tensor) -> bool:
    """False for tensors that torch's dispatch resolves before an operator reads them: batched
    ones (vmap, is_grads_batched), negated views, zeros without memory, tensors of another
    device.  Most of them are a plain torch.Tensor on a CUDA device by type."""
    return torch._C._dispatch_keys(t) == _PLAIN_KEYS


def _by_operator(do: Tensor, *saved: Tensor) -> bool:
    """torch.compile, make_fx / AOTAutograd (a dispatch mode is active), fake / meta tensors,
    or ones without values of their own: the backward is the registered operator, one node
    of the graph.  So it is under create_graph=True, the one time that grad mode is on here:
    the operator has no second derivative and refuses one, where gradients without a graph
    would leave it out of a sum in silence.  Otherwise, eager on the GPU, it is the same
    implementation without a second operator dispatch."""
    return (torch.is_grad_enabled() or torch.compiler.is_compiling() or torch._C._len_torch_dispatch_stack() > 0
            or type(do) is not torch.Tensor or not all(map(_holds_values, (do, *saved))))


def _backward(ctx, do, _dlse):
    q, k, v, o, lse = ctx.saved_tensors
    if do is None:
        return (None,) * (3 + len(ctx.rest))
    if _by_operator(do, q, k, v):
        dq, dk, dv = torch.ops.chia_attn.bwd(do, q, k, v, o, lse, *ctx.rest)
    else:
        from .attention import run_backward

        dq, dk, dv = run_backward(do, q, k, v, o, lse if lse.numel() else None, _params(*ctx.rest))
    return (dq, dk, dv) + (None,) * len(ctx.rest)


fwd.register_autograd(_backward, setup_context=_setup_context)


def _schema_args(params: dict) -> tuple:
    """attention()'s keyword parameters as the operators' trailing arguments (per-head
    vectors already float32 device tensors or None; scale None = default)."""
    return (params["norm"], bool(params["causal"]), int(params["window"] or 0), int(params["dilation"] or 1),
            int(params["block"] or 0), int(params["prefix"] or 0),
            None if params["scale"] is None else float(params["scale"]), params["head_scale"],
            params["alibi_slopes"], float(params["softcap"] or 0.0), float(params["bias"]),
            float(params["post_scale"]))


def call_fwd(q: Tensor, k: Tensor, v: Tensor, params: dict) -> Tuple[Tensor, Tensor]:
    """torch.ops.chia_attn.fwd with attention()'s keyword parameters."""
    return torch.ops.chia_attn.fwd(q, k, v, *_schema_args(params))


# ---- eager training ------------------------------------------------------------------
# The operators' dispatch (schema parsing, the autograd wrapper's pytree maps, one
# Python call per dispatch key) costs more host time than the rest of an eager
# training call together.  Plain CUDA tensors outside every mechanism that needs to
# see the operator take the same implementations through an autograd function of
# their own, which saves the tensors the registered formula saves.

_PLAIN_TYPES = (Tensor, torch.nn.Parameter)


def plain_eager(*tensors) -> bool:
    """True when the operator's dispatch would do nothing but call the implementation:
    plain CUDA tensors that hold their values, no dispatch or function mode (tracing,
    FakeTensor), no functorch transform (vmap, grad, jvp), no forward-mode level and no
    TorchScript tracing.  (A profiler's trace shows such a call as the autograd function
    below and not as chia_attn::fwd.)"""
    for t in tensors:
        if type(t) not in _PLAIN_TYPES or not _holds_values(t):
            return False
    return (torch._C._len_torch_dispatch_stack() == 0 and torch._C._len_torch_function_stack() == 0
            and not torch._C._are_functorch_transforms_active()
            and torch.autograd.forward_ad._current_level < 0 and torch._C._get_tracing_state() is None)


class _EagerAttention(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, k, v, *rest):
        from .attention import run_forward

        o, lse = run_forward(q, k, v, _params(*rest))
        ctx.rest = rest
        ctx.save_for_backward(q, k, v, o, lse)
        ctx.set_materialize_grads(False)
        return o

    @staticmethod
    def backward(ctx, do):
        return _backward(ctx, do, None)


def eager_fwd(q: Tensor, k: Tensor, v: Tensor, params: dict) -> Tensor:
    """call_fwd()'s o, differentiable, for plain_eager() tensors."""
    return _EagerAttention.apply(q, k, v, *_schema_args(params))


# ---- packed variable-length batches ------------------------------------------------
#   chia_attn::fwd_varlen(q, k, v, cu_seqlens, max_seqlen, <parameters>) -> (o, lse)
#       q, o [T, H, D]; k, v [T, H_kv, D]; lse float32 [T, H] (softmax) or [0]
#   chia_attn::bwd_varlen(do, q, k, v, o, lse, cu_seqlens, max_seqlen, <parameters>) -> (dq, dk, dv)
# max_seqlen <= 0: the longest sequence (read from cu_seqlens on the host).

def _max_len(max_seqlen: int):
    return None if max_seqlen <= 0 else max_seqlen


@torch.library.custom_op(f"{NAMESPACE}::fwd_varlen", mutates_args=(), device_types="cuda")
def fwd_varlen(q: Tensor, k: Tensor, v: Tensor, cu_seqlens: Tensor, max_seqlen: int, norm: str, causal: bool,
               window: int, dilation: int, block: int, prefix: int, scale: Optional[float],
               head_scale: Optional[Tensor], alibi_slopes: Optional[Tensor], softcap: float, bias: float,
               post_scale: float) -> Tuple[Tensor, Tensor]:
    from .attention import run_forward_varlen

    p = _params(norm, causal, window, dilation, block, prefix, scale, head_scale, alibi_slopes, softcap, bias,
                post_scale)
    return run_forward_varlen(q, k, v, cu_seqlens, _max_len(max_seqlen), p)


@fwd_varlen.register_fake
def _fwd_varlen_fake(q, k, v, cu_seqlens, max_seqlen, norm, causal, window, dilation, block, prefix, scale,
                     head_scale, alibi_slopes, softcap, bias, post_scale):
    torch._check(q.dim() == 3, lambda: "q must be 3-D [T, H, D]")
    T, H, _ = q.shape
    lse_shape = (T, H) if norm == "softmax" else (0, 0)
    return torch.empty_like(q, memory_format=torch.contiguous_format), q.new_empty(lse_shape, dtype=torch.float32)


@torch.library.custom_op(f"{NAMESPACE}::bwd_varlen", mutates_args=(), device_types="cuda")
def bwd_varlen(do: Tensor, q: Tensor, k: Tensor, v: Tensor, o: Tensor, lse: Tensor, cu_seqlens: Tensor,
               max_seqlen: int, norm: str, causal: bool, window: int, dilation: int, block: int, prefix: int,
               scale: Optional[float], head_scale: Optional[Tensor], alibi_slopes: Optional[Tensor], softcap: float,
               bias: float, post_scale: float) -> Tuple[Tensor, Tensor, Tensor]:
    from .attention import run_backward_varlen

    p = _params(norm, causal, window, dilation, block, prefix, scale, head_scale, alibi_slopes, softcap, bias,
                post_scale)
    return run_backward_varlen(do, q, k, v, o, lse, cu_seqlens, _max_len(max_seqlen), p)


@bwd_varlen.register_fake
def _bwd_varlen_fake(do, q, k, v, o, lse, cu_seqlens, max_seqlen, norm, causal, window, dilation, block, prefix,
                     scale, head_scale, alibi_slopes, softcap, bias, post_scale):
    return (torch.empty_like(q, memory_format=torch.contiguous_format),
            torch.empty_like(k, memory_format=torch.contiguous_format),
            torch.empty_like(v, memory_format=torch.contiguous_format))


def _setup_context_varlen(ctx, inputs, output):
    q, k, v, cu_seqlens, *rest = inputs
    o, lse = output
    ctx.rest = rest  # max_seqlen .. post_scale, schema order
    ctx.save_for_backward(q, k, v, o, lse, cu_seqlens)
    ctx.mark_non_differentiable(lse)
    ctx.set_materialize_grads(False)


def _backward_varlen(ctx, do, _dlse):
    q, k, v, o, lse, cu_seqlens = ctx.saved_tensors
    if do is None:
        return (None,) * (4 + len(ctx.rest))
    if _by_operator(do, q, k, v):
        dq, dk, dv = torch.ops.chia_attn.bwd_varlen(do, q, k, v, o, lse, cu_seqlens, *ctx.rest)
    else:
        from .attention import run_backward_varlen

        max_seqlen, *rest = ctx.rest
        dq, dk, dv = run_backward_varlen(do, q, k, v, o, lse, cu_seqlens, _max_len(max_seqlen), _params(*rest))
    return (dq, dk, dv) + (None,) * (1 + len(ctx.rest))


fwd_varlen.register_autograd(_backward_varlen, setup_context=_setup_context_varlen)


def call_fwd_varlen(q: Tensor, k: Tensor, v: Tensor, cu_seqlens: Tensor, max_seqlen: Optional[int],
                    params: dict) -> Tuple[Tensor, Tensor]:
    """torch.ops.chia_attn.fwd_varlen with attention_varlen()'s keyword parameters."""
    return torch.ops.chia_attn.fwd_varlen(q, k, v, cu_seqlens, int(max_seqlen or 0), *_schema_args(params))


class _EagerAttentionVarlen(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, k, v, cu_seqlens, max_seqlen, *rest):
        from .attention import run_forward_varlen

        o, lse = run_forward_varlen(q, k, v, cu_seqlens, _max_len(max_seqlen), _params(*rest))
        ctx.rest = (max_seqlen, *rest)
        ctx.save_for_backward(q, k, v, o, lse, cu_seqlens)
        ctx.set_materialize_grads(False)
        return o

    @staticmethod
    def backward(ctx, do):
        return _backward_varlen(ctx, do, None)


def eager_fwd_varlen(q: Tensor, k: Tensor, v: Tensor, cu_seqlens: Tensor, max_seqlen: Optional[int],
                     params: dict) -> Tensor:
    """call_fwd_varlen()'s o, differentiable, for plain_eager() tensors."""
    return _EagerAttentionVarlen.apply(q, k, v, cu_seqlens, int(max_seqlen or 0), *_schema_args(params))


# ---- FP8 forward -----------------------------------------------------------------

@torch.library.custom_op(f"{NAMESPACE}::fwd_fp8", mutates_args=(), device_types="cuda")
def fwd_fp8(q: Tensor, k: Tensor, v: Tensor, q_descale: float, k_descale: float, v_descale: float, norm: str,
            causal: bool, window: int, dilation: int, block: int, prefix: int, scale: Optional[float],
            head_scale: Optional[Tensor], alibi_slopes: Optional[Tensor], softcap: float, bias: float,
            post_scale: float) -> Tensor:
    from .attention import attention_fp8

    return attention_fp8(q, k, v, q_descale=q_descale, k_descale=k_descale, v_descale=v_descale,
                         **_params(norm, causal, window, dilation, block, prefix, scale, head_scale, alibi_slopes,
                                   softcap, bias, post_scale))


@fwd_fp8.register_fake
def _fwd_fp8_fake(q, k, v, q_descale, k_descale, v_descale, norm, causal, window, dilation, block, prefix, scale,
                  head_scale, alibi_slopes, softcap, bias, post_scale):
    torch._check(q.dim() == 4, lambda: "q must be 4-D [B, H, S, D]")
    return torch.empty(q.shape, dtype=torch.bfloat16, device=q.device)


def call_fwd_fp8(q: Tensor, k: Tensor, v: Tensor, q_descale: float, k_descale: float, v_descale: float,
                 params: dict) -> Tensor:
    """torch.ops.chia_attn.fwd_fp8 with attention_fp8()'s keyword parameters (per-head
    vectors float32 device tensors or None; scale None = default)."""
    return torch.ops.chia_attn.fwd_fp8(q, k, v, float(q_descale), float(k_descale), float(v_descale),
                                       params["norm"], bool(params["causal"]), int(params["window"] or 0),
                                       int(params["dilation"] or 1), int(params["block"] or 0),
                                       int(params["prefix"] or 0),
                                       None if params["scale"] is None else float(params["scale"]),
                                       params["head_scale"], params["alibi_slopes"],
                                       float(params["softcap"] or 0.0), float(params["bias"]),
                                       float(params["post_scale"]))
