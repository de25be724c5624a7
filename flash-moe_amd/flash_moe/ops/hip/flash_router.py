"""Product-key router op: top-k over the nk*nk pair sums of two per-token score vectors.

Same call signature, return values and argument checks as ``triton_flash_router_func``
(flash_moe/ops/triton/flash_router.py:381-382; contract docs/flash_router.md:16-40); the work is done
by ``fmoe_router_topk`` in libflashmoe_hip.so.
"""
from __future__ import annotations

from typing import Optional, Tuple

import torch

from flash_moe import _C
from flash_moe.ops.utils import ensure_contiguous


def router_topk_gates(
    router_logits: torch.Tensor,
    num_expert_keys: int,
    num_experts_per_tok: int,
    with_gates: bool = False,
    norm_topk_prob: bool = False,
) -> Tuple[torch.Tensor, torch.Tensor, Optional[torch.Tensor]]:
    """Launch the router kernel.  Returns ``(scores, indices, gates-or-None)``.

    ``gates = exp(scores)`` (divided by its per-token sum if ``norm_topk_prob``) is what
    FlashMoE.forward computes right after the router (flash_moe/modules/flash_moe.py:80-85); asking
    for it here saves two or three elementwise launches.
    """
    _check_topk_args(router_logits, num_expert_keys, num_experts_per_tok)
    return _C.native().router_topk(router_logits, num_expert_keys, num_experts_per_tok, with_gates, bool(norm_topk_prob))


def _check_topk_args(router_logits, num_expert_keys, num_experts_per_tok):
    # the three checks of _flash_router_forward (flash_router.py:257-263), same exception type
    assert router_logits.dim() == 3, (
        "router_logits must be a 3D tensor of shape (2, batch_size * seq_len, num_expert_keys)"
    )
    assert router_logits.size(0) == 2, "The first dimension of router_logits must be 2"
    assert 0 <= num_experts_per_tok <= num_expert_keys, (
        f"num_experts_per_tok should be in [0, {num_expert_keys}], but got {num_experts_per_tok}"
    )


def check_norm(norm: torch.nn.BatchNorm1d):
    """The batch-norm state the native calls take: ``(running_mean, running_var, num_batches_tracked, training, momentum, eps)``."""
    if norm.affine or norm.momentum is None or not norm.track_running_stats:
        raise ValueError("the fused router expects BatchNorm1d(affine=False, momentum=<float>, track_running_stats=True)")
    buffers = norm._buffers
    return (buffers["running_mean"], buffers["running_var"], buffers["num_batches_tracked"], norm.training, norm.momentum, norm.eps)


def check_router_args(tokens, gate_weight, norm, num_expert_keys, num_experts_per_tok, split_query=False):
    """Argument checks of the fused routing stage; returns ``check_norm(norm)``."""
    width = tokens.shape[1] // 2 if split_query else tokens.shape[1]
    if tokens.dim() != 2 or gate_weight.shape != (2 * num_expert_keys, width):
        raise ValueError("expected tokens [T, H] and a router gate weight [2*num_expert_keys, H] "
                         "([2*num_expert_keys, H/2] sub-key tables with split_query)")
    assert 0 <= num_experts_per_tok <= num_expert_keys, (
        f"num_experts_per_tok should be in [0, {num_expert_keys}], but got {num_experts_per_tok}"
    )
    if gate_weight.dtype != tokens.dtype:
        raise TypeError(f"router gate weight has dtype {gate_weight.dtype}, tokens have {tokens.dtype}")
    state = check_norm(norm)
    if norm.training and tokens.shape[0] == 1:
        raise ValueError(f"Expected more than 1 value per channel when training, got input size {tuple(tokens.shape)}")
    rm, rv = state[0], state[1]
    if not (rm.is_contiguous() and rv.is_contiguous() and rm.dtype == rv.dtype):
        raise ValueError("running statistics must be contiguous and of one dtype")
    return state


def router_forward(tokens: torch.Tensor, gate_weight: torch.Tensor, norm: torch.nn.BatchNorm1d, num_expert_keys: int,
                   num_experts_per_tok: int, norm_topk_prob: bool = False, return_logits32: bool = False,
                   return_stats: bool = False, split_query: bool = False):
    """The block's whole routing stage in one call of ``fmoe_router_forward``: batch-norm (training or evaluation
    mode, taken from ``norm.training``; its running statistics are updated in place), the router gate, the per-half
    log-softmax, the product-key top-k and the gates (flash_moe/modules/flash_moe.py:62-85).

    Returns ``(router_logits [T, 2*nk] in tokens.dtype, scores [T,K] fp32, indices [T,K] int64, gates [T,K] in
    tokens.dtype)``, plus the fp32 logits the routing was computed from when ``return_logits32`` is set, plus the
    batch-norm mean and 1/sqrt(var + eps) used ([2*H] fp32, a view of the call's workspace) when ``return_stats`` is set.
    ``split_query``: ``gate_weight`` is two sub-key tables [2*nk, H/2], each scoring its own half of the normalised query
    (``fmoe_router_forward_split``; equal to a block-diagonal [2*nk, H] gate); the module never uses this form.
    """
    state = check_router_args(tokens, gate_weight, norm, num_expert_keys, num_experts_per_tok, split_query)
    logits, scores, indices, gates, logits32, stats = _C.native().router_forward(
        tokens, gate_weight, *state, num_expert_keys, num_experts_per_tok, bool(norm_topk_prob), split_query)
    result = (logits, scores, indices, gates)
    if return_logits32:
        result += (logits32,)
    if return_stats:
        result += (stats,)
    return result


def router_prologue_backward(dlogits32: torch.Tensor, tokens: torch.Tensor, gate_weight: torch.Tensor, stats: torch.Tensor,
                             training: bool):
    """``(dtokens, dgate_weight)`` of ``logits = BatchNorm1d(tokens) @ gate_weight.T`` from the fp32 gradient of the logits
    [T, 2*nk] and the forward's batch-norm statistics ``stats`` ([2*H] fp32: mean, 1/sqrt(var + eps));
    ``fmoe_router_prologue_backward``."""
    return _C.native().router_prologue_backward(dlogits32, tokens, gate_weight, stats, training)


def route_backward(dgates: torch.Tensor, indices: torch.Tensor, logits32: torch.Tensor, num_expert_keys: int,
                   norm_topk_prob: bool = False, dlogits: torch.Tensor = None) -> torch.Tensor:
    """Gradient of the fp32 gate logits [T, 2*nk] from the gradient of the gates [T, K] (``fmoe_route_backward``): the
    backward of per-half log-softmax, product-key top-k, exp and optional renormalisation
    (flash_moe/modules/flash_moe.py:69-85) in one launch.  ``dlogits`` ([T, 2*nk] in the gates' dtype), the gradient of the
    router logits the block returns, is added when given."""
    return _C.native().route_backward(dgates, indices, logits32, num_expert_keys, bool(norm_topk_prob), dlogits)


def router_prologue(tokens: torch.Tensor, gate_weight: torch.Tensor, norm: torch.nn.BatchNorm1d):
    """Differentiable router prologue ``logits = BatchNorm1d(x) @ gate_weight.T`` (flash_moe/modules/flash_moe.py:62-67):
    ``(logits_fp32 [T, 2*nk], logits [T, 2*nk] in tokens.dtype)``, the fp32 logits the routing is computed from and their rounding
    to the activation dtype.  Forward: the batch-norm and gate launches of ``fmoe_router_forward`` (top_k = 0); backward:
    ``fmoe_router_prologue_backward``.  ``norm``'s running statistics are updated in training mode, as by any forward."""
    state = check_router_args(tokens, gate_weight, norm, gate_weight.shape[0] // 2, 0)
    return _C.native().router_prologue(tokens, gate_weight, *state)


def router_topk_backward(dscores: torch.Tensor, indices: torch.Tensor, num_expert_keys: int) -> torch.Tensor:
    """Scatter of ``dscores`` [T, K] onto the two halves' keys -> [2, T, nk] in ``dscores.dtype`` (``fmoe_router_topk_backward``):
    each selected pair's gradient goes to its two keys (flash_moe/ops/triton/flash_router.py:317-344)."""
    return _C.native().router_topk_backward(dscores, indices, num_expert_keys)


def flash_router_func(router_logits, num_expert_keys, num_experts_per_tok):
    """router_logits [2, T, nk] -> scores [T, K] (dtype of the input), indices [T, K] int64."""
    _check_topk_args(router_logits, num_expert_keys, num_experts_per_tok)
    return _C.native().router_func(router_logits, num_expert_keys, num_experts_per_tok)


class FlashRouterFunc(torch.autograd.Function):
    """``flash_router_func`` as an autograd function under the reference's class name (flash_moe/ops/triton/flash_router.py:347),
    for callers that apply or subclass it; the op itself takes the native node."""

    @staticmethod
    @ensure_contiguous
    def forward(ctx, router_logits, num_expert_keys, num_experts_per_tok):
        scores, indices, _ = router_topk_gates(router_logits, num_expert_keys, num_experts_per_tok)
        ctx.mark_non_differentiable(indices)
        ctx.save_for_backward(indices)
        ctx.num_expert_keys = num_expert_keys
        return scores, indices

    @staticmethod
    @ensure_contiguous
    def backward(ctx, dscores, dindices):
        (indices,) = ctx.saved_tensors
        return router_topk_backward(dscores, indices, ctx.num_expert_keys), None, None


class RouterPrologueFunc(torch.autograd.Function):
    """``router_prologue`` as an autograd function."""

    @staticmethod
    def forward(ctx, tokens, gate_weight, norm):
        logits, _, _, _, logits32, stats = router_forward(tokens, gate_weight, norm, gate_weight.shape[0] // 2, 0,
                                                          return_logits32=True, return_stats=True)
        ctx.save_for_backward(tokens, gate_weight, stats.clone())
        ctx.training = norm.training
        return logits32, logits

    @staticmethod
    def backward(ctx, dlogits32, dlogits):
        tokens, gate_weight, stats = ctx.saved_tensors
        return (*router_prologue_backward(dlogits32 + dlogits.float(), tokens, gate_weight, stats, ctx.training), None)
