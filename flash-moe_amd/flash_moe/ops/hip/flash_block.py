"""The whole FlashMoE block forward as one call of ``fmoe_block_forward``.

``block_forward`` computes what FlashMoE.forward computes on the flattened tokens
(flash_moe/modules/flash_moe.py:55-105): router -> routed experts -> shared SwiGLU MLP + add.  The routing
(logits, expert ids, gates, statistics) is that of ``router_forward`` to the last bit, and the output that of calling
``expert_forward`` and ``mlp_forward(residual=...)`` with it; for at most 2048 tokens, where stages share launches, the MLP's
fp32 sums may be taken in another order, beyond that the output is the same to the last bit too.  The single call keeps
every intermediate in one workspace and skips the conversion of expert ids to table offsets.
"""
from __future__ import annotations

import torch

from flash_moe import _C
from flash_moe.ops.hip.flash_router import check_norm


def block_forward(tokens: torch.Tensor, gate_proj: torch.Tensor, up_proj: torch.Tensor, down_proj: torch.Tensor,
                  router_gate: torch.Tensor, norm: torch.nn.BatchNorm1d, down_embed: torch.Tensor, up_embed: torch.Tensor,
                  num_expert_keys: int, num_experts_per_tok: int, norm_topk_prob: bool = False,
                  return_routing: bool = False):
    """tokens [T, H] -> ``(out [T, H], router_logits [T, 2*nk])`` in tokens.dtype, plus ``(indices int64, gates)``
    [T, K] when ``return_routing`` is set.  ``norm.training`` selects batch or running statistics; the running
    statistics are updated in place in training mode."""
    out, logits, *routing = block(tokens, gate_proj, up_proj, down_proj, router_gate, norm, down_embed, up_embed, num_expert_keys,
                                  num_experts_per_tok, norm_topk_prob, return_routing=return_routing)
    return (out, logits.transpose(0, 1).reshape(tokens.shape[0], 2 * num_expert_keys), *routing)


def block(hidden_states, gate_proj, up_proj, down_proj, router_gate, norm, down_embed, up_embed, num_expert_keys,
          num_experts_per_tok, norm_topk_prob=False, differentiable=False, return_routing=False):
    """``[out, router_logits]`` as the module returns them: ``out`` in the shape of ``hidden_states`` [..., H], the logits
    [2, T, nk] (a token's two halves side by side in memory).  ``differentiable``: when one of the inputs
    requires a gradient, one autograd node whose forward is
    ``fmoe_block_forward_save`` and whose backward is ``fmoe_block_backward``, with gradients for the tokens and every weight.
    The reference reaches the same gradients through autograd of its eager ops around the three Triton functions
    (flash_moe/modules/flash_moe.py:55-105)."""
    assert 0 <= num_experts_per_tok <= num_expert_keys, (
        f"num_experts_per_tok should be in [0, {num_expert_keys}], but got {num_experts_per_tok}"
    )
    return _C.native().block(hidden_states, gate_proj, up_proj, down_proj, router_gate, down_embed, up_embed, *check_norm(norm),
                             num_expert_keys, num_experts_per_tok, norm_topk_prob, differentiable, return_routing)
