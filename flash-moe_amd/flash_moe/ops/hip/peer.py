"""PEER op: ``out[t] = sum_k gelu(<x_t, Wd[idx[t,k]]>) * w[t,k] * Wu[idx[t,k]]`` (erf GELU).

Same call signature and return value as ``triton_peer_func`` (flash_moe/ops/triton/peer.py:246-255; note the
argument order: routing weights before indices); the work is done by ``fmoe_peer_forward`` in libflashmoe_hip.so,
which runs the routed-expert kernels with GELU in place of SiLU.  Forward only, as in the reference (peer.py:241-243).
"""
from __future__ import annotations

from flash_moe import _C


def peer_func(hidden_states, down_embed, up_embed, routing_weights, indices):
    return _C.native().peer_func(hidden_states, down_embed, up_embed, routing_weights, indices)


class PEERFunc:
    """The op under the reference's class name (flash_moe/ops/triton/peer.py:222); its backward raises there as well."""

    apply = staticmethod(peer_func)
