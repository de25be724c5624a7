// The whole FlashMoE block forward in one call: router -> routed experts -> shared SwiGLU MLP (+ add).
// The stages are the same launches as the per-op entry points; what the single call adds is that intermediates never
// leave the caller's one workspace, the router writes the experts' table-row offsets directly (no int64 -> offset
// pass), and the host does one FFI call instead of three plus their allocations.
#include "fmoe_common.h"

namespace fmoe {
namespace {

struct BlockPlan {
    size_t off_router, off_logits32, off_scores, off_indices, off_gates, off_expert, off_act, off_experts_out, off_sums, bytes;
    SmallPlan small;
};

BlockPlan plan_block(int64_t T_, int H, int I, int nk, int64_t E, int K, int dtype) {
    BlockPlan p;
    const size_t elt = dtype_size(dtype);
    size_t o = 0;
    auto take = [&](size_t n) { const size_t at = o; o = round_up(o + n, 256); return at; };
    p.off_router = take(fmoe_router_workspace_bytes(T_, H, nk));
    p.off_logits32 = take((size_t)T_ * 2 * nk * 4);
    p.off_scores = take((size_t)T_ * K * 4);
    p.off_indices = take((size_t)T_ * K * 8);
    p.off_gates = take((size_t)T_ * K * elt);
    p.off_expert = take(fmoe_expert_workspace_bytes(T_, H, E, K, dtype));
    p.off_act = take(fmoe_mlp_workspace_bytes(T_, H, I, dtype));
    p.off_experts_out = take((size_t)T_ * H * elt);
    p.small = plan_small(T_, H, I, nk, E, K, dtype);
    p.off_sums = take(p.small.sums_bytes);
    p.bytes = o;
    return p;
}

}  // namespace
}  // namespace fmoe

extern "C" size_t fmoe_block_workspace_bytes(int64_t num_tokens, int hidden, int intermediate, int num_keys,
                                             int64_t num_experts, int top_k, int dtype) {
    if (num_tokens <= 0 || hidden <= 0 || intermediate <= 0 || num_keys <= 0 || num_experts <= 0 || top_k < 0 ||
        !fmoe::dtype_ok(dtype))
        return 0;
    return fmoe::plan_block(num_tokens, hidden, intermediate, num_keys, num_experts, top_k, dtype).bytes;
}

namespace fmoe {
namespace {

// What a training forward leaves for the backward, in one caller-owned buffer.
struct SavedPlan {
    size_t off_logits32, off_indices, off_gates, off_stats, off_products, off_experts, bytes;
};

SavedPlan plan_saved(int64_t T_, int H, int I, int nk, int64_t E, int K, int dtype) {
    SavedPlan p;
    const size_t elt = dtype_size(dtype);
    size_t o = 0;
    auto take = [&](size_t n) { const size_t at = o; o = round_up(o + n, 256); return at; };
    p.off_logits32 = take((size_t)T_ * 2 * nk * 4);
    p.off_indices = take((size_t)T_ * K * 8);
    p.off_gates = take((size_t)T_ * K * elt);
    p.off_stats = take((size_t)2 * H * 4);
    p.off_products = take((size_t)2 * T_ * I * elt);
    p.off_experts = take(fmoe_expert_saved_bytes(T_, H, E, K, dtype));
    p.bytes = o;
    return p;
}

struct BlockBackwardPlan {
    size_t off_dgates, off_dlogits32, off_dx_experts, off_planes, off_stage, stage_bytes, bytes;
    MlpBackwardPlan mlp;
    PrologueBackwardPlan prologue;
};

// The stages run one after the other on one stream, so they share one scratch area, but for the MLP's slices of k: the last stage adds
// those of its dx.
BlockBackwardPlan plan_block_backward(int64_t T_, int H, int I, int nk, int64_t E, int K, int dtype) {
    BlockBackwardPlan p;
    const size_t elt = dtype_size(dtype);
    size_t o = 0;
    auto take = [&](size_t n) { const size_t at = o; o = round_up(o + n, 256); return at; };
    p.off_dgates = take((size_t)T_ * K * elt);
    p.off_dlogits32 = take(route_backward_prepares(nk, K) ? 0 : (size_t)T_ * 2 * nk * 4);
    p.off_dx_experts = take((size_t)T_ * H * elt);
    p.mlp = plan_mlp_backward(T_, H, I, dtype, true);
    p.prologue = plan_prologue_backward(T_, H, nk, dtype);
    p.off_planes = take(p.mlp.part_bytes > 0 ? p.mlp.part_bytes : 256);
    p.stage_bytes = p.mlp.off_part;
    const size_t experts = fmoe_expert_backward_workspace_bytes(T_, H, E, K, dtype);
    if (experts > p.stage_bytes) p.stage_bytes = experts;
    if (p.prologue.bytes > p.stage_bytes) p.stage_bytes = p.prologue.bytes;
    p.off_stage = take(p.stage_bytes);
    p.bytes = o;
    return p;
}

int check_block(const char* who, int64_t num_tokens, int hidden, int intermediate, int64_t num_experts, int num_keys, int top_k,
                int dtype) {
    FMOE_REQUIRE(dtype_ok(dtype), FMOE_ERR_BAD_DTYPE, "%s: unknown dtype %d", who, dtype);
    FMOE_REQUIRE(num_tokens >= 0 && hidden > 0 && intermediate > 0 && num_experts > 0 && num_keys > 0, FMOE_ERR_BAD_SHAPE,
                 "%s: bad shape T=%lld H=%d I=%d E=%lld nk=%d", who, (long long)num_tokens, hidden, intermediate,
                 (long long)num_experts, num_keys);
    FMOE_REQUIRE((int64_t)num_keys * num_keys <= num_experts, FMOE_ERR_BAD_SHAPE,
                 "%s: num_keys^2 = %lld exceeds num_experts = %lld", who, (long long)num_keys * num_keys, (long long)num_experts);
    FMOE_REQUIRE(top_k >= 0 && top_k <= num_keys, FMOE_ERR_TOPK_RANGE, "num_experts_per_tok should be in [0, %d], but got %d",
                 num_keys, top_k);
    return FMOE_OK;
}

// saved: the buffer of a training forward, or NULL
int block_forward_impl(const char* who, const void* x, const void* gate_proj_w, const void* up_proj_w, const void* down_proj_w,
                       const void* router_gate_w, const void* down_embed, const void* up_embed, void* running_mean,
                       void* running_var, int64_t* num_batches_tracked, int stats_dtype, int training, float momentum, float eps,
                       int64_t num_tokens, int hidden, int intermediate, int64_t num_experts, int num_keys, int top_k, int dtype,
                       int norm_topk_prob, void* out, void* router_logits, int64_t* indices_out, void* gates_out, char* saved,
                       void* workspace, size_t workspace_bytes, void* stream) {
    if (int rc = check_block(who, num_tokens, hidden, intermediate, num_experts, num_keys, top_k, dtype)) return rc;
    if (num_tokens == 0) return FMOE_OK;
    FMOE_REQUIRE(x && gate_proj_w && up_proj_w && down_proj_w && router_gate_w && down_embed && up_embed && out && router_logits,
                 FMOE_ERR_NULL_POINTER, "%s: null tensor pointer", who);
    // what the stages would refuse is refused here, before the first launch
    const int vec = (int)(16 / dtype_size(dtype));
    FMOE_REQUIRE(hidden % vec == 0 && (dtype == FMOE_F32 || intermediate % 8 == 0), FMOE_ERR_ALIGNMENT,
                 "%s: hidden=%d and intermediate=%d must give 16-byte rows", who, hidden, intermediate);
    FMOE_REQUIRE(aligned16(x) && aligned16(gate_proj_w) && aligned16(up_proj_w) && aligned16(down_proj_w) &&
                     aligned16(router_gate_w) && aligned16(down_embed) && aligned16(up_embed) && aligned16(out),
                 FMOE_ERR_ALIGNMENT, "%s: tensor pointers must be 16-byte aligned", who);
    FMOE_REQUIRE(num_tokens < (1ll << 31) && num_experts < (1ll << 31), FMOE_ERR_UNSUPPORTED,
                 "%s: T=%lld or E=%lld >= 2^31", who, (long long)num_tokens, (long long)num_experts);
    const BlockPlan p = plan_block(num_tokens, hidden, intermediate, num_keys, num_experts, top_k, dtype);
    FMOE_REQUIRE(workspace && workspace_bytes >= p.bytes && aligned16(workspace), FMOE_ERR_WORKSPACE,
                 "%s: workspace of %zu bytes needed, %zu given", who, p.bytes, workspace_bytes);
    hipStream_t s = (hipStream_t)stream;
    char* ws = (char*)workspace;
    float* logits32 = (float*)(ws + p.off_logits32);
    float* scores = (float*)(ws + p.off_scores);
    int64_t* indices = indices_out ? indices_out : (int64_t*)(ws + p.off_indices);
    void* gates = gates_out ? gates_out : (void*)(ws + p.off_gates);
    float* stats = nullptr;
    void* products = nullptr;
    void* act = ws + p.off_act;
    void* expert_saved = nullptr;
    if (saved != nullptr) {
        const SavedPlan sp = plan_saved(num_tokens, hidden, intermediate, num_keys, num_experts, top_k, dtype);
        expert_saved = saved + sp.off_experts;
        logits32 = (float*)(saved + sp.off_logits32);
        indices = (int64_t*)(saved + sp.off_indices);
        gates = saved + sp.off_gates;
        stats = (float*)(saved + sp.off_stats);
        products = saved + sp.off_products;
    }
    void* expert_ws = ws + p.off_expert;
    void* experts = ws + p.off_experts_out;
    const size_t elt = dtype_size(dtype);

    const bool slices = expert_slices_usable(num_tokens, hidden, num_experts, top_k, dtype);
    uint32_t* offsets = slices ? expert_workspace_offsets(expert_ws) : nullptr;
    float* expert_scores = nullptr;
    if (slices && expert_saved != nullptr) {
        const ExpertSaved kept = expert_saved_plan(num_tokens, hidden, num_experts, top_k, dtype).at(expert_saved);
        offsets = kept.off32;
        expert_scores = kept.scores;
    }
    auto gate_up = [&]() {
        return products ? fmoe_mlp_gate_up_save(x, gate_proj_w, up_proj_w, num_tokens, hidden, intermediate, dtype, act, products, stream)
                        : fmoe_mlp_gate_up(x, gate_proj_w, up_proj_w, num_tokens, hidden, intermediate, dtype, act, stream);
    };
    // The statistics a call lacks, and the shapes the router refuses, are reported by the router's own entry
    const bool up_beside = p.small.gate_and_up && dtype_ok(stats_dtype) &&
                           (training ? num_tokens > 1 : running_mean != nullptr && running_var != nullptr);
    const bool down_beside = p.small.select_and_down;
    int rc;
    if (up_beside) {
        float* scratch = (float*)(ws + p.off_router);
        rc = small_gate_and_up(x, gate_proj_w, up_proj_w, router_gate_w, running_mean, running_var, num_batches_tracked, stats_dtype, training,
                               momentum, eps, num_tokens, hidden, intermediate, num_keys, dtype, router_logits, logits32, act, products,
                               scratch, stats ? stats : scratch + router_block_stats_bytes(hidden) / sizeof(float), s);
        if (rc == FMOE_OK && !down_beside && top_k > 0)
            rc = launch_router_from_logits(logits32, num_tokens, num_keys, top_k, scores, indices, gates, dtype, norm_topk_prob, offsets,
                                           (uint32_t)(hidden * elt), s);
    } else {
        rc = router_forward_impl(x, router_gate_w, running_mean, running_var, num_batches_tracked, stats_dtype, training, momentum, eps,
                                 num_tokens, hidden, num_keys, down_beside ? 0 : top_k, dtype, norm_topk_prob, router_logits, logits32, scores,
                                 indices, gates, offsets, (uint32_t)(hidden * elt), ws + p.off_router, p.off_logits32 - p.off_router, s, 0, 0,
                                 stats);
    }
    if (rc) return rc;
    if (down_beside) {
        if (!up_beside)
            if ((rc = gate_up())) return rc;
        return small_select_down_experts(x, down_proj_w, down_embed, up_embed, num_tokens, hidden, intermediate, num_experts, num_keys, top_k,
                                         dtype, norm_topk_prob, out, logits32, scores, indices, gates, act, (float*)(ws + p.off_sums), s);
    }
    const void* residual = nullptr;
    if (top_k > 0) {
        if (slices)
            rc = expert_slices_prepared(x, down_embed, up_embed, gates, num_tokens, hidden, num_experts, top_k, dtype, experts,
                                        expert_ws, offsets, expert_scores, s);
        else if (expert_saved != nullptr)
            rc = fmoe_expert_forward_save(x, down_embed, up_embed, indices, gates, num_tokens, hidden, num_experts, top_k, dtype, experts,
                                          expert_saved, fmoe_expert_saved_bytes(num_tokens, hidden, num_experts, top_k, dtype), expert_ws,
                                          p.off_act - p.off_expert, stream);
        else
            rc = fmoe_expert_forward(x, down_embed, up_embed, indices, gates, num_tokens, hidden, num_experts, top_k, dtype,
                                     experts, expert_ws, p.off_act - p.off_expert, stream);
        if (rc) return rc;
        residual = experts;
    }
    if (!up_beside)
        if ((rc = gate_up())) return rc;
    const size_t act_bytes = fmoe_mlp_workspace_bytes(num_tokens, hidden, intermediate, dtype);
    const size_t planes = fmoe_mlp_down_workspace_bytes(num_tokens, hidden, intermediate, dtype);
    return fmoe_mlp_down_ws(act, down_proj_w, num_tokens, hidden, intermediate, dtype, residual, out, ws + p.off_act + (act_bytes - planes), planes,
                            stream);
}

}  // namespace
}  // namespace fmoe

extern "C" int fmoe_block_forward(const void* x, const void* gate_proj_w, const void* up_proj_w, const void* down_proj_w,
                                  const void* router_gate_w, const void* down_embed, const void* up_embed,
                                  void* running_mean, void* running_var, int64_t* num_batches_tracked, int stats_dtype,
                                  int training, float momentum, float eps, int64_t num_tokens, int hidden,
                                  int intermediate, int64_t num_experts, int num_keys, int top_k, int dtype,
                                  int norm_topk_prob, void* out, void* router_logits, int64_t* indices_out,
                                  void* gates_out, void* workspace, size_t workspace_bytes, void* stream) {
    fmoe::clear_error();
    return fmoe::block_forward_impl("fmoe_block_forward", x, gate_proj_w, up_proj_w, down_proj_w, router_gate_w, down_embed, up_embed,
                                    running_mean, running_var, num_batches_tracked, stats_dtype, training, momentum, eps, num_tokens,
                                    hidden, intermediate, num_experts, num_keys, top_k, dtype, norm_topk_prob, out, router_logits,
                                    indices_out, gates_out, nullptr, workspace, workspace_bytes, stream);
}

extern "C" size_t fmoe_block_saved_bytes(int64_t num_tokens, int hidden, int intermediate, int num_keys, int64_t num_experts,
                                         int top_k, int dtype) {
    if (num_tokens <= 0 || hidden <= 0 || intermediate <= 0 || num_keys <= 0 || num_experts <= 0 || top_k <= 0 || !fmoe::dtype_ok(dtype))
        return 0;
    return fmoe::plan_saved(num_tokens, hidden, intermediate, num_keys, num_experts, top_k, dtype).bytes;
}

extern "C" int fmoe_block_forward_save(const void* x, const void* gate_proj_w, const void* up_proj_w, const void* down_proj_w,
                                       const void* router_gate_w, const void* down_embed, const void* up_embed,
                                       void* running_mean, void* running_var, int64_t* num_batches_tracked, int stats_dtype,
                                       int training, float momentum, float eps, int64_t num_tokens, int hidden,
                                       int intermediate, int64_t num_experts, int num_keys, int top_k, int dtype,
                                       int norm_topk_prob, void* out, void* router_logits, void* saved, size_t saved_bytes,
                                       void* workspace, size_t workspace_bytes, void* stream) {
    using namespace fmoe;
    clear_error();
    const size_t need = fmoe_block_saved_bytes(num_tokens, hidden, intermediate, num_keys, num_experts, top_k, dtype);
    FMOE_REQUIRE(num_tokens == 0 || top_k > 0, FMOE_ERR_UNSUPPORTED, "fmoe_block_forward_save: top_k = 0 keeps nothing for a backward pass");
    FMOE_REQUIRE(num_tokens == 0 || (saved && saved_bytes >= need && aligned16(saved)), FMOE_ERR_WORKSPACE,
                 "fmoe_block_forward_save: buffer of %zu bytes needed, %zu given", need, saved_bytes);
    return block_forward_impl("fmoe_block_forward_save", x, gate_proj_w, up_proj_w, down_proj_w, router_gate_w, down_embed, up_embed,
                              running_mean, running_var, num_batches_tracked, stats_dtype, training, momentum, eps, num_tokens,
                              hidden, intermediate, num_experts, num_keys, top_k, dtype, norm_topk_prob, out, router_logits, nullptr,
                              nullptr, (char*)saved, workspace, workspace_bytes, stream);
}

extern "C" size_t fmoe_block_backward_workspace_bytes(int64_t num_tokens, int hidden, int intermediate, int num_keys,
                                                      int64_t num_experts, int top_k, int dtype) {
    if (num_tokens <= 0 || hidden <= 0 || intermediate <= 0 || num_keys <= 0 || num_experts <= 0 || top_k <= 0 || !fmoe::dtype_ok(dtype))
        return 0;
    return fmoe::plan_block_backward(num_tokens, hidden, intermediate, num_keys, num_experts, top_k, dtype).bytes;
}

extern "C" int fmoe_block_backward(const void* dout, const void* dlogits, const void* x, const void* gate_proj_w,
                                   const void* up_proj_w, const void* down_proj_w, const void* router_gate_w,
                                   const void* down_embed, const void* up_embed, const void* saved, int training,
                                   int64_t num_tokens, int hidden, int intermediate, int64_t num_experts, int num_keys, int top_k,
                                   int dtype, int norm_topk_prob, void* dx, void* dgate_proj_w, void* dup_proj_w,
                                   void* ddown_proj_w, void* drouter_gate_w, void* ddown_embed, void* dup_embed, void* workspace,
                                   size_t workspace_bytes, void* stream) {
    using namespace fmoe;
    clear_error();
    if (int rc = check_block("fmoe_block_backward", num_tokens, hidden, intermediate, num_experts, num_keys, top_k, dtype)) return rc;
    FMOE_REQUIRE(num_tokens > 0 && top_k > 0, FMOE_ERR_UNSUPPORTED, "fmoe_block_backward: needs at least one token and one expert per token");
    FMOE_REQUIRE(dout && saved && dx, FMOE_ERR_NULL_POINTER, "fmoe_block_backward: null tensor pointer");
    const BlockBackwardPlan p = plan_block_backward(num_tokens, hidden, intermediate, num_keys, num_experts, top_k, dtype);
    FMOE_REQUIRE(workspace && workspace_bytes >= p.bytes && aligned16(workspace), FMOE_ERR_WORKSPACE,
                 "fmoe_block_backward: workspace of %zu bytes needed, %zu given", p.bytes, workspace_bytes);
    const SavedPlan sp = plan_saved(num_tokens, hidden, intermediate, num_keys, num_experts, top_k, dtype);
    const char* sv = (const char*)saved;
    const float* logits32 = (const float*)(sv + sp.off_logits32);
    const int64_t* indices = (const int64_t*)(sv + sp.off_indices);
    char* ws = (char*)workspace;
    void *dgates = ws + p.off_dgates, *dx_experts = ws + p.off_dx_experts, *stage = ws + p.off_stage;
    float* dlogits32 = (float*)(ws + p.off_dlogits32);
    KeptPlanes kept = {};
    int rc = mlp_backward_impl(dout, x, gate_proj_w, up_proj_w, down_proj_w, sv + sp.off_products, num_tokens, hidden, intermediate, dtype, dx,
                               dgate_proj_w, dup_proj_w, ddown_proj_w, p.mlp, stage, p.stage_bytes, ws + p.off_planes, &kept, (hipStream_t)stream);
    if (rc) return rc;
    rc = fmoe_expert_backward_saved(dout, x, down_embed, up_embed, indices, sv + sp.off_gates, sv + sp.off_experts, num_tokens, hidden,
                                    num_experts, top_k, dtype, dx_experts, ddown_embed, dup_embed, dgates, stage, p.stage_bytes, stream);
    if (rc) return rc;
    const float* mean_rstd = (const float*)(sv + sp.off_stats);
    const bool prepares = route_backward_prepares(num_keys, top_k);
    const PrologueOperands operands = prologue_operands(x, mean_rstd, hidden, p.prologue, stage);
    rc = route_backward_impl(dgates, indices, logits32, dlogits, num_keys, num_tokens * num_keys, num_tokens, num_keys, top_k, dtype,
                             norm_topk_prob, dlogits32, (hipStream_t)stream, prepares ? &operands : nullptr);
    if (rc) return rc;
    // the three token gradients are summed where the last of them is formed
    return router_prologue_backward_impl(dlogits32, x, router_gate_w, mean_rstd, training, num_tokens, hidden,
                                         num_keys, dtype, dx, drouter_gate_w, {kept.planes ? nullptr : dx, dx_experts, kept.planes, kept.slices}, p.prologue,
                                         stage, p.stage_bytes, (hipStream_t)stream, prepares);
}
