"""Causal self-attention on the gfx950 MFMA kernels (src/reversibility/model.py:26-45).

The reference's ``CausalSelfAttention`` projects to a packed ``qkv`` of width
``3 d``, views it as ``[B, T, 3, H, hd]``, permutes it into three strided
``[B, H, T, hd]`` tensors for ``F.scaled_dot_product_attention(is_causal=True)``,
and transposes the result back to ``[B, T, d]`` for the output projection;
autograd then stacks ``dq, dk, dv`` back into the packed layout.  Here the
kernels read ``qkv`` in the layout the qkv GEMM wrote, write the output in the
layout the output GEMM reads, and write the gradient straight into a packed
``dqkv`` (``rv_attn_fwd`` / ``rv_attn_bwd``, csrc/attention.hip): no permute,
transpose or concatenation copies.  Forward keeps the base-2 log-sum-exp per
query; backward is deterministic (no atomics).

``enable_attention(model)`` patches every block's ``attn.forward``; calls the
kernels do not cover (no fp16 ``qkv`` -- i.e. not under fp16 autocast --, head
sizes other than 32/64/128, dropout in training mode, CPU tensors) keep the
reference computation, recorded in ``paths.report()`` (or raising under
``paths.strict()``).
"""
from __future__ import annotations

import types

import torch
import torch.nn.functional as F
from torch.autograd.function import once_differentiable

from . import linear as _linear
from . import paths
from ._hip import RV_F16, RV_F32, _check, _stream, library
from .mlp import cast_operands, splitk_workspace

HEAD_DIMS = (32, 64, 128)


def supported(qkv: torch.Tensor, heads: int, dropout: float = 0.0) -> bool:
    if not (qkv.is_cuda and qkv.dtype == torch.float16 and qkv.ndim == 3 and dropout == 0.0):
        return False
    width = qkv.shape[-1]
    return width % (3 * heads) == 0 and width // (3 * heads) in HEAD_DIMS


class CausalAttention(torch.autograd.Function):
    """``qkv`` fp16 ``[B, T, 3 d]`` -> causal attention output fp16 ``[B, T, d]``."""

    @staticmethod
    def forward(ctx, qkv, heads):
        batch, seq, width = qkv.shape
        d = width // 3
        qkv = qkv.contiguous()
        out = torch.empty(batch, seq, d, device=qkv.device, dtype=torch.float16)
        lse = torch.empty(batch * heads, seq, device=qkv.device, dtype=torch.float32)
        _check(library().rv_attn_fwd(qkv.data_ptr(), batch, seq, heads, d // heads,
                                     out.data_ptr(), lse.data_ptr(), _stream(qkv)), "rv_attn_fwd")
        ctx.save_for_backward(qkv, out, lse)
        ctx.heads = heads
        return out

    @staticmethod
    @once_differentiable
    def backward(ctx, dout):
        qkv, out, lse = ctx.saved_tensors
        batch, seq, width = qkv.shape
        heads = ctx.heads
        lib = library()
        dout = dout.to(torch.float16).contiguous()
        dqkv = torch.empty_like(qkv)
        nbytes = lib.rv_attn_bwd_workspace_bytes(batch, seq, heads)
        if nbytes < 0:
            _check(-nbytes, "rv_attn_bwd_workspace_bytes")
        ws = torch.empty(nbytes // 4, device=qkv.device, dtype=torch.float32)
        _check(lib.rv_attn_bwd(qkv.data_ptr(), out.data_ptr(), dout.data_ptr(), lse.data_ptr(),
                               batch, seq, heads, width // 3 // heads, dqkv.data_ptr(),
                               ws.data_ptr(), nbytes, _stream(qkv)), "rv_attn_bwd")
        return dqkv, None


class AttentionLayer(torch.autograd.Function):
    """``proj(causal_attention(qkv(x)))`` of one layer under fp16 autocast as one
    autograd node: the same kernels on the same values as ``FusedLinear``,
    ``CausalAttention`` and ``FusedLinear`` in turn, with one launch for the
    operand casts and one for the two weight gradients (reduced over the
    rows in another fixed order than each alone).  The weights' fp16 casts live
    from forward to backward (2 bytes per weight), and qkv, its log-sum-exp and the
    attention output to the end of the backward, where three nodes free them one
    after the other (8 bytes per token and column more at the input gradient)."""

    @staticmethod
    def forward(ctx, x, w_qkv, w_proj, heads):
        batch, seq, d = x.shape
        rows, out_f = batch * seq, w_proj.shape[0]
        lib, st = library(), _stream(x)
        x16, qkv16, proj16 = cast_operands(x.reshape(rows, d).contiguous(), w_qkv, w_proj)
        dev = x.device
        qkv = torch.empty(rows, 3 * d, device=dev, dtype=torch.float16)
        mixed = torch.empty(rows, d, device=dev, dtype=torch.float16)
        lse = torch.empty(batch * heads, seq, device=dev, dtype=torch.float32)
        y = torch.empty(batch, seq, out_f, device=dev, dtype=torch.float16)
        ws, nbytes = splitk_workspace(x16, rows, 3 * d, d)
        _check(lib.rv_linear_fwd_ws(x16.data_ptr(), d, qkv16.data_ptr(), rows, d, 3 * d,
                                    qkv.data_ptr(), ws.data_ptr() if nbytes else None, nbytes,
                                    st), "rv_linear_fwd")
        _check(lib.rv_attn_fwd(qkv.data_ptr(), batch, seq, heads, d // heads, mixed.data_ptr(),
                               lse.data_ptr(), st), "rv_attn_fwd")
        ws, nbytes = splitk_workspace(x16, rows, out_f, d)
        _check(lib.rv_linear_fwd_ws(mixed.data_ptr(), d, proj16.data_ptr(), rows, d, out_f,
                                    y.data_ptr(), ws.data_ptr() if nbytes else None, nbytes, st),
               "rv_linear_fwd")
        ctx.save_for_backward(x16, w_qkv, w_proj, qkv16, proj16, qkv, mixed, lse)
        ctx.heads, ctx.x_dtype, ctx.shape = heads, x.dtype, (batch, seq, d)
        return y

    @staticmethod
    @once_differentiable
    def backward(ctx, gradient):
        x16, w_qkv, w_proj, qkv16, proj16, qkv, mixed, lse = ctx.saved_tensors
        (batch, seq, d), heads, out_f = ctx.shape, ctx.heads, w_proj.shape[0]
        rows = batch * seq
        lib, st, dev = library(), _stream(x16), x16.device
        dy = gradient.reshape(rows, out_f).to(torch.float16).contiguous()
        dx = dw_qkv = dw_proj = None
        need_x, need_qkv, need_proj = ctx.needs_input_grad[:3]
        if need_x or need_qkv:
            dmixed = torch.empty_like(mixed)
            ws, nbytes = splitk_workspace(dy, rows, d, out_f)
            _check(lib.rv_linear_dx_ws(dy.data_ptr(), proj16.data_ptr(), rows, d, out_f,
                                       dmixed.data_ptr(), RV_F16, ws.data_ptr() if nbytes else None,
                                       nbytes, st), "rv_linear_dx")
            dqkv = torch.empty_like(qkv)
            nbytes = lib.rv_attn_bwd_workspace_bytes(batch, seq, heads)
            if nbytes < 0:
                _check(-nbytes, "rv_attn_bwd_workspace_bytes")
            ws = torch.empty(nbytes // 4, device=dev, dtype=torch.float32)
            _check(lib.rv_attn_bwd(qkv.data_ptr(), mixed.data_ptr(), dmixed.data_ptr(), lse.data_ptr(),
                                   batch, seq, heads, d // heads, dqkv.data_ptr(), ws.data_ptr(),
                                   nbytes, st), "rv_attn_bwd")
            del dmixed, ws  # free for the buffers below
        if need_x:
            dx = torch.empty(batch, seq, d, device=dev, dtype=ctx.x_dtype)
            ws, nbytes = splitk_workspace(dqkv, rows, d, 3 * d)
            code = RV_F32 if ctx.x_dtype == torch.float32 else RV_F16
            _check(lib.rv_linear_dx_ws(dqkv.data_ptr(), qkv16.data_ptr(), rows, d, 3 * d,
                                       dx.data_ptr(), code, ws.data_ptr() if nbytes else None,
                                       nbytes, st), "rv_linear_dx")
        if need_qkv and need_proj:
            dw_qkv, dw_proj = torch.empty_like(w_qkv), torch.empty_like(w_proj)
            nbytes = lib.rv_linear_dw_pair_workspace_bytes(rows, d, 3 * d, d, out_f)
            if nbytes < 0:
                _check(-nbytes, "rv_linear_dw_pair_workspace_bytes")
            ws = torch.empty(nbytes // 4, device=dev, dtype=torch.float32) if nbytes else None
            _check(lib.rv_linear_dw_pair(
                dqkv.data_ptr(), x16.data_ptr(), d, 3 * d, dw_qkv.data_ptr(), dy.data_ptr(),
                mixed.data_ptr(), d, out_f, dw_proj.data_ptr(), rows, 0,
                ws.data_ptr() if nbytes else None, nbytes, st), "rv_linear_dw_pair")
        elif need_qkv:  # the other projection is frozen
            dw_qkv = _linear.weight_grad(dqkv.view(rows, 3 * d), x16, w_qkv)
        elif need_proj:
            dw_proj = _linear.weight_grad(dy, mixed, w_proj)
        return dx, dw_qkv, dw_proj, None


def _layer_supported(attn: torch.nn.Module, x: torch.Tensor, dropout: float) -> bool:
    """Whether ``AttentionLayer`` is what the layer's own modules would compute
    on their kernels, one after the other."""
    qkv, proj = attn.qkv, attn.proj
    return (x.ndim == 3 and x.numel() > 0 and dropout == 0.0 and _linear.plain_layer(qkv)
            and _linear.plain_layer(proj)
            and _linear.supported(x, qkv.weight, None) and proj.weight.is_cuda
            and proj.weight.dtype == torch.float32 and proj.weight.is_contiguous()
            and proj.weight.shape[0] % 128 == 0 and proj.weight.shape[1] == x.shape[-1]
            and qkv.weight.shape[0] == 3 * x.shape[-1] and x.shape[-1] % attn.n_heads == 0
            and x.shape[-1] // attn.n_heads in HEAD_DIMS)


def causal_attention(qkv: torch.Tensor, heads: int) -> torch.Tensor:
    """Causal attention of a packed fp16 ``qkv`` on the kernels; raises on inputs
    they do not cover."""
    if not supported(qkv, heads):
        raise ValueError("fused attention needs a CUDA fp16 qkv [B, T, 3 d] with head size "
                         f"in {HEAD_DIMS}")
    return CausalAttention.apply(qkv, heads)


def reference_attention(qkv: torch.Tensor, heads: int, dropout: float = 0.0) -> torch.Tensor:
    """The reference's computation (model.py:40-45) on a packed ``qkv``."""
    batch, length, width = qkv.shape
    d = width // 3
    q, k, v = qkv.view(batch, length, 3, heads, d // heads).permute(2, 0, 3, 1, 4).unbind(0)
    mixed = F.scaled_dot_product_attention(q, k, v, dropout_p=dropout, is_causal=True)
    return mixed.transpose(1, 2).reshape(batch, length, d)


def enable_attention(model: torch.nn.Module) -> None:
    """Route every block's attention through the fused kernels where they apply."""
    def forward(attn, x):
        dropout = attn.dropout if attn.training else 0.0
        if _layer_supported(attn, x, dropout):
            paths.took("linear", "mfma")
            paths.took("attention", "hip")
            paths.took("linear", "mfma")
            return AttentionLayer.apply(x, attn.qkv.weight, attn.proj.weight, attn.n_heads)
        qkv = attn.qkv(x)
        if supported(qkv, attn.n_heads, dropout):
            paths.took("attention", "hip")
            mixed = CausalAttention.apply(qkv, attn.n_heads)
        else:
            paths.took("attention", "sdpa",
                       f"attention kernels need a CUDA fp16 qkv, head size in {HEAD_DIMS} and no "
                       f"dropout (got {qkv.dtype} on {qkv.device.type}, head size "
                       f"{qkv.shape[-1] // (3 * attn.n_heads)}, dropout {dropout})")
            mixed = reference_attention(qkv, attn.n_heads, dropout)
        return attn.proj(mixed)
    for block in model.blocks:
        block.attn.forward = types.MethodType(forward, block.attn)
