"""Shared SwiGLU MLP op: ``(silu(x Wg^T) * (x Wu^T)) Wd^T``.

Same call signature and return value as ``triton_flash_mlp_func``
(flash_moe/ops/triton/flash_mlp.py:169-181); the work is done by ``fmoe_mlp_forward`` in
libflashmoe_hip.so (two MFMA GEMMs, the activation fused into the first one's epilogue).
"""
from __future__ import annotations

from typing import Optional

import torch

from flash_moe import _C
from flash_moe.ops.utils import ensure_contiguous


def mlp_forward(x, gate_weight, up_weight, down_weight, residual: Optional[torch.Tensor] = None) -> torch.Tensor:
    """``x`` may have any leading shape; the last dimension is the hidden size.  ``residual`` (same shape
    as the output) is added in the second GEMM's epilogue (the add of flash_moe/modules/flash_moe.py:101)."""
    return _C.native().mlp_forward(x, gate_weight, up_weight, down_weight, residual)


def mlp_forward_saving(x, gate_weight, up_weight, down_weight, residual: Optional[torch.Tensor] = None):
    """``mlp_forward`` that also returns the [2, T, I] gate and up products for ``mlp_backward`` (``fmoe_mlp_gate_up_save``
    then ``fmoe_mlp_down``), as the reference's SwiGLU function saves them (flash_moe/ops/triton/flash_mlp.py:153-159)."""
    return _C.native().mlp_forward_saving(x, gate_weight, up_weight, down_weight, residual)


def mlp_backward(dout, x, gate_weight, up_weight, down_weight, saved=None):
    """Gradients ``(dx, dgate_weight, dup_weight, ddown_weight)`` of ``mlp_forward`` without residual
    (``fmoe_mlp_backward``): the gate and up products come from ``saved`` (``mlp_forward_saving``) or are recomputed, the
    SwiGLU gradient is the fused kernel behind ``swiglu_backward``.  The gradients of the gate and up weights are the two
    halves of one buffer."""
    return _C.native().mlp_backward(dout, x, gate_weight, up_weight, down_weight, saved)


def swiglu_backward(a: torch.Tensor, b: torch.Tensor, dc: torch.Tensor):
    """``(da, db)`` for ``c = silu(a) * b`` (``fmoe_swiglu_backward``; flash_moe/ops/triton/flash_mlp.py:126-150)."""
    return _C.native().swiglu_backward(a, b, dc)


def flash_mlp_func(x: torch.Tensor, gate_weight: torch.Tensor, up_weight: torch.Tensor, down_weight: torch.Tensor) -> torch.Tensor:
    return _C.native().mlp_func(x, gate_weight, up_weight, down_weight)


class FlashMLPFunc(torch.autograd.Function):
    """``flash_mlp_func`` as an autograd function, for callers that apply or subclass it; the op itself takes the native node."""

    @staticmethod
    @ensure_contiguous
    def forward(ctx, x, gate_weight, up_weight, down_weight):
        if x.numel() == 0 or not any(ctx.needs_input_grad):
            ctx.save_for_backward(x, gate_weight, up_weight, down_weight)
            return mlp_forward(x, gate_weight, up_weight, down_weight)
        out, saved = mlp_forward_saving(x, gate_weight, up_weight, down_weight)
        ctx.save_for_backward(x, gate_weight, up_weight, down_weight, saved)
        return out

    @staticmethod
    @ensure_contiguous
    def backward(ctx, dout):
        return mlp_backward(dout, *ctx.saved_tensors)
