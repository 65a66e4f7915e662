"""Fused cross-entropy and SwiGLU on gfx950, behind the reference's operator surface.

``TiledCrossEntropy`` / ``cross_entropy_sum`` mirror src/reversibility/kernels.py:56-85:
``apply(logits, labels)`` takes contiguous ``[tokens, vocab]`` fp16/fp32 logits
and int64 labels on the same device and returns the summed loss (fp32); rows
labelled -100 contribute nothing.  It keeps the reference's Half-logsoftmax ->
fp32 NLL policy: the log-probability at the target is rounded to the logits
dtype before it is negated and summed, and the backward rounds the
log-probability again before the exponential.  One HIP kernel reads each row
once per pass (rv_ce_fwd / rv_ce_bwd).

``FusedSwiGLU`` / ``enable_swiglu`` mirror src/reversibility/kernels.py:113-138:
``apply(up)`` takes the packed up-projection ``[..., 2W]`` (gate = first W
columns, value = last W), returns ``[..., W]`` in the input dtype, and its
backward returns the packed gradient.  Same ValueError contract (contiguous
CUDA FP16/FP32, even final width; no CPU fallback).  Rounding points follow
the reference: silu is rounded to the I/O dtype before the multiply, and
``dy * value`` before the sigmoid-derivative product.
"""
from __future__ import annotations

import types

import torch
from torch.autograd.function import once_differentiable

from . import paths
from ._hip import ops


IGNORE_INDEX = -100


class TiledCrossEntropy(torch.autograd.Function):
    """Summed cross-entropy over vocabulary rows (kernels.py:56-80)."""

    @staticmethod
    def forward(ctx, logits, labels):
        if logits.device.type != "cuda" or logits.dtype not in (torch.float16, torch.float32):
            raise ValueError("Fused CE requires CUDA (ROCm device) FP16/FP32 logits; "
                             "no silent fallback")
        if (logits.ndim != 2 or not logits.is_contiguous() or labels.device != logits.device
                or labels.dtype != torch.int64 or labels.numel() != logits.shape[0]):
            raise ValueError("Contiguous [tokens,vocab] logits and matching CUDA int64 labels "
                             "required")
        labels = labels.contiguous()
        row_max, row_lse, losses = ops.ce_fwd(logits, labels, IGNORE_INDEX)
        ctx.save_for_backward(logits, labels, row_max, row_lse)
        return losses.sum()

    @staticmethod
    @once_differentiable
    def backward(ctx, gradient):
        logits, labels, row_max, row_lse = ctx.saved_tensors
        grad = gradient.detach().to(torch.float32).reshape(1).contiguous()
        return ops.ce_bwd(logits, labels, row_max, row_lse, grad, IGNORE_INDEX), None


def cross_entropy_sum(logits, labels):
    """Sum of per-token cross-entropy losses (kernels.py:83-84)."""
    return TiledCrossEntropy.apply(logits, labels)


VOCAB_ALIGN = 64  # padded logits row stride (in elements) of tied_head_ce
# widest row rv_ce_fused keeps in registers (32 16-byte vectors per thread)
FUSED_CE_MAX_COLS = 65536


def tied_head_ce(x16: torch.Tensor, head16: torch.Tensor, vocab: int, labels: torch.Tensor,
                 grad: torch.Tensor, dx_out: torch.Tensor | None = None,
                 dw_out: torch.Tensor | None = None, accumulate: bool = False):
    """One chunk of the tied head and its summed cross-entropy, forward and
    backward, with the logits stored at a padded row stride.

    The same computation as ``cross_entropy_sum(F.linear(x16, head16[:vocab]),
    labels)`` under fp16 autocast followed by its backward with upstream
    gradient ``grad`` (a device fp32 scalar): logits = fp16(x16 W^T); loss and
    dlogits from one pass of rv_ce_fused over each logits row (the two-pass
    rv_ce_fwd / rv_ce_bwd above FUSED_CE_MAX_COLS, same bits); dx = dlogits W and
    dW = dlogits^T x16 (fp16, as autocast's linear produces them).  The logits and
    the two gradients run on the MFMA kernels or on torch's GEMMs (``head_routes``,
    and operands off a 16-byte boundary; ``paths.report()`` has the sides taken,
    "mfma", "hipblaslt" or the logits' and the gradients').  ``head16`` is the fp16
    head with its rows padded to a multiple of VOCAB_ALIGN (as ``padded_head`` makes
    it), so every logits row starts 16-byte aligned.  Returns (loss sum, dx16, dW16
    [vocab, d]); dx16 is written into ``dx_out`` (contiguous fp16 [rows, d]) when
    given, and dW -- the same fp16 values widened -- into ``dw_out`` (contiguous fp32
    [vocab, d]; added to it with ``accumulate``), which is then returned for dW16.
    """
    rows, d = x16.shape
    padded = head16.shape[0]
    if (x16.dtype != torch.float16 or head16.dtype != torch.float16 or not x16.is_contiguous()
            or not head16.is_contiguous() or head16.shape[1] != d or padded % VOCAB_ALIGN
            or not 0 < vocab <= padded or labels.dtype != torch.int64
            or labels.numel() != rows or not x16.is_cuda):
        raise ValueError("tied_head_ce needs contiguous CUDA fp16 x [rows, d], a padded fp16 "
                         "head [padded, d] and int64 labels [rows]")
    # the kernels take raw pointers: memory of another device would fault there
    if any(t is not None and t.device != x16.device for t in (head16, labels, grad, dx_out)):
        raise ValueError("tied_head_ce needs its head, labels, gradient and dx_out on x's device")
    if dw_out is not None and (dw_out.dtype != torch.float32 or not dw_out.is_contiguous()
                               or tuple(dw_out.shape) != (vocab, d)
                               or dw_out.device != x16.device):
        raise ValueError("tied_head_ce's dw_out must be a contiguous fp32 [vocab, d] tensor on "
                         "x's device")
    from ._hip import RV_F16, RV_F32, _check, _stream, library
    lib = library()
    labels = labels.contiguous()
    own_logits, own_grads = head_routes(rows, d, padded)
    aligned = x16.data_ptr() % 16 == 0 and head16.data_ptr() % 16 == 0
    own_logits = own_logits and aligned
    own_grads = (own_grads and aligned and (dw_out is None or dw_out.data_ptr() % 16 == 0)
                 and (dx_out is None or (dx_out.dtype == torch.float16 and dx_out.is_contiguous()
                                         and dx_out.shape == x16.shape
                                         and dx_out.data_ptr() % 16 == 0)))
    sides = ["mfma" if own else "hipblaslt" for own in (own_logits, own_grads)]
    paths.took("tied_head", "fused-ce+" + "/".join(dict.fromkeys(sides)))
    if own_logits:
        logits = torch.empty(rows, padded, device=x16.device, dtype=torch.float16)
        _check(lib.rv_head_logits(x16.data_ptr(), head16.data_ptr(), rows, d, vocab, padded,
                                  logits.data_ptr(), _stream(x16)), "rv_head_logits")
    else:
        logits = torch.mm(x16, head16.t())                   # [rows, padded] fp16
        if own_grads and vocab < padded:
            logits[:, vocab:].zero_()  # rv_head_dx reads the pad columns
    rmax, rlse, losses = (torch.empty(rows, device=x16.device, dtype=torch.float32)
                          for _ in range(3))
    st = _stream(x16)
    if rows and vocab <= FUSED_CE_MAX_COLS:
        # one pass: loss and gradient, written over the logits
        dlogits = logits
        _check(lib.rv_ce_fused(logits.data_ptr(), RV_F16, padded, labels.data_ptr(), rows, vocab,
                               IGNORE_INDEX, grad.data_ptr(), rmax.data_ptr(), rlse.data_ptr(),
                               losses.data_ptr(), dlogits.data_ptr(), st), "rv_ce_fused")
    else:
        dlogits = torch.empty_like(logits)
        if own_grads:
            dlogits[:, vocab:].zero_()  # rv_head_dx reads the pad columns
        if rows:
            _check(lib.rv_ce_fwd(logits.data_ptr(), RV_F16, padded, labels.data_ptr(), rows,
                                 vocab, IGNORE_INDEX, rmax.data_ptr(), rlse.data_ptr(),
                                 losses.data_ptr(), st), "rv_ce_fwd")
            _check(lib.rv_ce_bwd(logits.data_ptr(), RV_F16, padded, labels.data_ptr(),
                                 rmax.data_ptr(), rlse.data_ptr(), grad.data_ptr(), rows, vocab,
                                 IGNORE_INDEX, dlogits.data_ptr(), st), "rv_ce_bwd")
    del logits
    if own_grads:
        nbytes = lib.rv_head_workspace_bytes(rows, d, vocab, padded)
        if nbytes < 0:
            _check(-nbytes, "rv_head_workspace_bytes")
        ws = torch.empty(nbytes // 4, device=x16.device, dtype=torch.float32) if nbytes else None
        ws_ptr = ws.data_ptr() if nbytes else None
        dx16 = dx_out if dx_out is not None else torch.empty_like(x16)
        _check(lib.rv_head_dx(dlogits.data_ptr(), head16.data_ptr(), rows, d, vocab, padded,
                              dx16.data_ptr(), ws_ptr, nbytes, st), "rv_head_dx")
        dw = dw_out if dw_out is not None else torch.empty(vocab, d, device=x16.device,
                                                           dtype=torch.float16)
        _check(lib.rv_head_dw(dlogits.data_ptr(), x16.data_ptr(), rows, d, vocab, padded,
                              dw.data_ptr(), RV_F16 if dw_out is None else RV_F32,
                              int(accumulate and dw_out is not None), ws_ptr, nbytes, st),
               "rv_head_dw")
        return losses.sum(), dx16, dw
    d_view = dlogits[:, :vocab]
    if dx_out is not None:
        dx16 = torch.mm(d_view, head16[:vocab], out=dx_out)
    else:
        dx16 = torch.mm(d_view, head16[:vocab])
    dw16 = torch.mm(d_view.t(), x16)
    if dw_out is None:
        return losses.sum(), dx16, dw16
    if accumulate:
        dw_out.add_(dw16)
    else:
        dw_out.copy_(dw16)
    return losses.sum(), dx16, dw_out


def head_routes(rows: int, d: int, padded: int) -> tuple[bool, bool]:
    """Which of the head's products take the MFMA kernels: (logits, gradients).
    They need a width that is a multiple of 128 and a 256-row tile of the logits
    within 2 GiB; within that, the side that is faster (us, own / torch's GEMM,
    operands evicted before each product; widths 128 .. 1024, 64 .. 32768 rows,
    vocabularies 1000 .. 50257):

    logits     up to width 512, and at any below one round of 256 x 256 tiles:
               16896 x 256 over 50257 619 / 607, over 10007 149 / 291, 8192 x 512 over
               50257 498 / 542.  Over a longer reduction the library's tile is the
               better one: 32768 x 1024 over 50257 3227 / 2878, 8192 x 768 over
               32000 448 / 372
    gradients  all but width 384 above 8192 rows, where the 128-column tiles read
               the logits three times: 24000 x 384 over 32000 1665 / 1228 (dx and dW
               together); 16896 x 256 over 50257 852 / 1069, 32768 x 1024 5592 / 5976,
               24000 x 640 over 32000 2123 / 2963, 12288 x 896 1676 / 1727
    """
    if rows <= 0 or d % 128 or 512 * padded >= (1 << 31) - (1 << 24):
        return False, False
    tiles = -(-rows // 256) * -(-padded // 256)
    return d <= 512 or tiles <= 256, d != 384 or rows <= 8192


def padded_head(weight: torch.Tensor) -> torch.Tensor:
    """fp16 copy of a [vocab, d] head with zero rows up to a multiple of VOCAB_ALIGN."""
    vocab, d = weight.shape
    padded = -(-vocab // VOCAB_ALIGN) * VOCAB_ALIGN
    head = torch.empty(padded, d, device=weight.device, dtype=torch.float16)
    head[:vocab].copy_(weight)
    head[vocab:].zero_()
    return head


def _validate(up: torch.Tensor) -> None:
    # kernels.py:116-117
    if (up.device.type != "cuda" or up.dtype not in (torch.float16, torch.float32)
            or not up.is_contiguous() or up.shape[-1] % 2):
        raise ValueError("Fused SwiGLU requires contiguous CUDA (ROCm device) FP16/FP32 "
                         "and even final width")


class FusedSwiGLU(torch.autograd.Function):
    """``silu(gate) * value`` over a packed ``[..., 2W]`` tensor."""

    @staticmethod
    def forward(ctx, up):
        _validate(up)
        output = ops.swiglu_fwd(up)
        ctx.save_for_backward(up)
        return output

    @staticmethod
    @once_differentiable
    def backward(ctx, gradient):
        up, = ctx.saved_tensors
        return ops.swiglu_bwd(up, gradient.contiguous())


def enable_swiglu(model: torch.nn.Module) -> None:
    """Patch every block's MLP to ``down(FusedSwiGLU(up(x)))`` (kernels.py:134-138)."""
    def forward(mlp, x):
        return mlp.down(FusedSwiGLU.apply(mlp.up(x)))
    for block in model.blocks:
        block.mlp.forward = types.MethodType(forward, block.mlp)
