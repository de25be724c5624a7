"""PEER op: ``out[t] = sum_k gelu(<x_t, Wd[idx[t,k]]>) * w[t,k] * Wu[idx[t,k]]`` (erf GELU).

Same call signature and return value as ``triton_peer_func`` (flash_moe/ops/triton/peer.py:246-255; note the
argument order: routing weights before indices); the work is done by ``fmoe_peer_forward`` in libflashmoe_hip.so,
which runs the routed-expert kernels with GELU in place of SiLU.  Forward only, as in the reference (peer.py:241-243).
"""
from __future__ import annotations

import torch

from flash_moe import _C
from flash_moe.ops.utils import ensure_contiguous


def peer_forward(hidden_states, down_embed, up_embed, routing_weights, indices) -> torch.Tensor:
    return _C.native().peer_forward(hidden_states, down_embed, up_embed, routing_weights, indices)


def peer_func(hidden_states, down_embed, up_embed, routing_weights, indices):
    return _C.native().peer_func(hidden_states, down_embed, up_embed, routing_weights, indices)


class PEERFunc(torch.autograd.Function):
    """The op as an autograd function under the reference's class name (flash_moe/ops/triton/peer.py:222); its backward raises there
    as well."""

    @staticmethod
    @ensure_contiguous
    def forward(ctx, hidden_states, down_embed, up_embed, routing_weights, indices):
        return peer_forward(hidden_states, down_embed, up_embed, routing_weights, indices)

    @staticmethod
    def backward(ctx, grad_output):
        raise NotImplementedError("PEER backward is not implemented (nor is it in the reference)")
