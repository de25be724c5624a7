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
from flash_moe.ops.hip.flash_expert import expert_backward, expert_forward
from flash_moe.ops.hip.flash_mlp import mlp_backward, mlp_forward_saving
from flash_moe.ops.hip.flash_router import check_norm, check_router_args, route_backward, router_forward, router_prologue_backward


def block_forward(tokens: torch.Tensor, gate_proj: torch.Tensor, up_proj: torch.Tensor, down_proj: torch.Tensor,
                  router_gate: torch.Tensor, norm: torch.nn.BatchNorm1d, down_embed: torch.Tensor, up_embed: torch.Tensor,
                  num_expert_keys: int, num_experts_per_tok: int, norm_topk_prob: bool = False,
                  return_routing: bool = False):
    """tokens [T, H] -> ``(out [T, H], router_logits [T, 2*nk])`` in tokens.dtype, plus ``(indices int64, gates)``
    [T, K] when ``return_routing`` is set.  ``norm.training`` selects batch or running statistics; the running
    statistics are updated in place in training mode."""
    check_router_args(tokens, router_gate, norm, num_expert_keys, num_experts_per_tok)      # tokens are 2-D here, unlike in block()
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


class FlashMoEBlockFunc(torch.autograd.Function):
    """The block with gradients for the tokens and every weight as an autograd function over the per-op calls: ``(out [T, H],
    router_logits [T, 2*nk])``, for callers that apply or subclass it; ``block`` takes the native node, one library call each way."""

    @staticmethod
    def forward(ctx, tokens, gate_proj, up_proj, down_proj, router_gate, down_embed, up_embed, norm, num_expert_keys,
                num_experts_per_tok, norm_topk_prob):
        x = tokens.contiguous()
        logits, _, indices, gates, logits32, stats = router_forward(
            x, router_gate, norm, num_expert_keys, num_experts_per_tok, norm_topk_prob, return_logits32=True, return_stats=True)
        experts = expert_forward(x, down_embed, up_embed, indices, gates)
        out, products = mlp_forward_saving(x, gate_proj, up_proj, down_proj, residual=experts)
        ctx.save_for_backward(x, gate_proj, up_proj, down_proj, router_gate, down_embed, up_embed, indices, gates, logits32,
                              stats.clone(), products)
        ctx.training, ctx.num_expert_keys, ctx.norm_topk_prob = norm.training, num_expert_keys, norm_topk_prob
        return out, logits

    @staticmethod
    def backward(ctx, dout, dlogits):
        x, wg, wu, wd, wr, ed, eu, indices, gates, logits32, stats, products = ctx.saved_tensors
        dx, dwg, dwu, dwd = mlp_backward(dout, x, wg, wu, wd, products)
        dx_experts, ded, deu, dgates = expert_backward(dout, x, ed, eu, indices, gates)
        dlogits32 = route_backward(dgates, indices, logits32, ctx.num_expert_keys, ctx.norm_topk_prob, dlogits)
        dx_router, dwr = router_prologue_backward(dlogits32, x, wr, stats, ctx.training)
        return dx.add_(dx_experts).add_(dx_router), dwg, dwu, dwd, dwr, ded, deu, None, None, None, None


def block_forward_autograd(tokens, gate_proj, up_proj, down_proj, router_gate, norm, down_embed, up_embed, num_expert_keys,
                           num_experts_per_tok, norm_topk_prob=False):
    """Differentiable ``block_forward``: ``(out [T, H], router_logits [T, 2*nk])``."""
    return FlashMoEBlockFunc.apply(tokens, gate_proj, up_proj, down_proj, router_gate, down_embed, up_embed, norm,
                                   num_expert_keys, num_experts_per_tok, norm_topk_prob)
