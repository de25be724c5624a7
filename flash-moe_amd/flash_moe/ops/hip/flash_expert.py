"""Routed-expert op: ``out[t] = sum_k silu(<x_t, Wd[idx[t,k]]>) * g[t,k] * Wu[idx[t,k]]``.

Same call signature and return value as ``triton_flash_expert_func``
(flash_moe/ops/triton/flash_expert.py:831-836; contract docs/flash_expert.md:17-58); the work is done
by ``fmoe_expert_forward`` in libflashmoe_hip.so.
"""
from __future__ import annotations

import torch

from flash_moe import _C
from flash_moe.ops.utils import ensure_contiguous


def expert_forward(hidden_states, down_weights, up_weights, indices, routing_weights, algo: int = _C.EXPERT_AUTO) -> torch.Tensor:
    """``algo`` picks the schedule (``_C.EXPERT_AUTO`` / ``EXPERT_ROWS`` / ``EXPERT_SLICES``); the result is the same."""
    return _C.native().expert_forward(hidden_states, down_weights, up_weights, indices, routing_weights, algo)


def expert_bucketing(indices: torch.Tensor, num_experts: int):
    """Expert-centric grouping of the (token, k) pairs on the GPU (``fmoe_expert_bucket``): returns
    ``(sorted_token_ids, expert_offsets, sorted_pair_ids, sorted_expert_ids)``, all int32; the first three are what
    ``_preprocess_expert_centric_indices_pytorch`` of the reference computes with sort / bincount / cumsum
    (flash_moe/ops/triton/flash_expert.py:528-577).  Pairs of expert ``e`` occupy slots ``[offsets[e], offsets[e+1])`` in
    ascending flattened position; ids outside ``[0, num_experts)`` are left out, so the three per-slot tensors have
    ``T*K`` entries of which the first ``offsets[-1]`` are meaningful.  No host synchronisation."""
    return _C.native().expert_bucketing(indices, num_experts)


def preprocess_expert_centric_indices(indices: torch.Tensor, routing_weights: torch.Tensor, num_experts: int):
    """Same return tuple as the reference's ``_preprocess_expert_centric_indices_pytorch(Indices, G, num_experts)``
    (flash_moe/ops/triton/flash_expert.py:528-577): ``(sorted_token_ids, sorted_G, expert_offsets, max_pairs_per_expert,
    sorted_pair_ids)``, for callers written against it.  ``max_pairs_per_expert`` is a host integer, so this helper
    synchronises like the reference does; the library's own forward and backward never need it.  Every id must lie in
    ``[0, num_experts)`` (the reference's contract)."""
    sorted_tokens, offsets, sorted_pairs, _ = expert_bucketing(indices, num_experts)
    sorted_g = routing_weights.reshape(-1)[sorted_pairs.long()]
    max_pairs = int((offsets[1:] - offsets[:-1]).max().item()) if num_experts > 0 else 0
    return sorted_tokens, sorted_g, offsets, max_pairs, sorted_pairs


def expert_backward(dexperts_states, hidden_states, down_weights, up_weights, indices, routing_weights):
    """Gradients ``(dhidden_states, ddown_weights, dup_weights, drouting_weights)`` of ``expert_forward``
    (``fmoe_expert_backward``; the reference's _flash_expert_backward, flash_moe/ops/triton/flash_expert.py:654-745).
    Deterministic; the scores are recomputed rather than saved."""
    return _C.native().expert_backward(dexperts_states, hidden_states, down_weights, up_weights, indices, routing_weights)


def flash_expert_func(hidden_states, down_weights, up_weights, indices, routing_weights):
    return _C.native().expert_func(hidden_states, down_weights, up_weights, indices, routing_weights)


class FlashExpertFunc(torch.autograd.Function):
    """``flash_expert_func`` as an autograd function under the reference's class name (flash_moe/ops/triton/flash_expert.py:748), for
    callers that apply or subclass it; the op itself takes the native node, which keeps the scores as well."""

    @staticmethod
    @ensure_contiguous
    def forward(ctx, hidden_states, down_weights, up_weights, indices, routing_weights):
        ctx.save_for_backward(hidden_states, down_weights, up_weights, indices, routing_weights)
        return expert_forward(hidden_states, down_weights, up_weights, indices, routing_weights)

    @staticmethod
    @ensure_contiguous
    def backward(ctx, dexperts_states):
        dx, dwd, dwu, dg = expert_backward(dexperts_states, *ctx.saved_tensors)
        return dx, dwd, dwu, None, dg
