"""Product-key-memory value lookup: ``out[t] = sum_k w[t,k] * values[idx[t,k]]``.

Same call signature and return value as ``triton_pkm_func`` (flash_moe/ops/triton/pkm.py:195-200); the work is done
by ``fmoe_pkm_forward`` in libflashmoe_hip.so (the second phase of the routed-expert kernels, with the routing weight as
the coefficient).  Forward only, as in the reference (pkm.py:190-192).
"""
from __future__ import annotations

import torch

from flash_moe import _C
from flash_moe.ops.utils import ensure_contiguous


def pkm_forward(values, routing_weights, indices) -> torch.Tensor:
    return _C.native().pkm_forward(values, routing_weights, indices)


def pkm_func(values, routing_weights, indices):
    return _C.native().pkm_func(values, routing_weights, indices)


class PKMFunc(torch.autograd.Function):
    """The op as an autograd function under the reference's class name (flash_moe/ops/triton/pkm.py:177); its backward raises there
    as well."""

    @staticmethod
    @ensure_contiguous
    def forward(ctx, values, routing_weights, indices):
        return pkm_forward(values, routing_weights, indices)

    @staticmethod
    def backward(ctx, grad_output):
        raise NotImplementedError("PKM backward is not implemented (nor is it in the reference)")
