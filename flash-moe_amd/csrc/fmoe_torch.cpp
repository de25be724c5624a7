// Torch binding of the FlashMoE library: argument checks, output and workspace allocation, the current stream and the autograd
// nodes, natively.  One Python call per op; everything below it (a training step makes 13 to 25 launches and a dozen
// allocations) runs without the interpreter, and the backward without the GIL.  The kernels are reached through the C ABI
// (include/flashmoe_hip.h) only.
//
// Why native: with ctypes calls and Python autograd functions the host side of one training step of the block took 520 us
// whatever the shapes, more than the GPU's 320 us at 615 tokens; a forward call took 39 us.
#include <ATen/hip/HIPContext.h>
#include <c10/hip/HIPStream.h>
#include <torch/extension.h>

#include "../../include/flashmoe_hip.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;
using OptTensor = std::optional<Tensor>;

int dtype_code(at::ScalarType t) {
    switch (t) {
        case at::kFloat: return FMOE_F32;
        case at::kBFloat16: return FMOE_BF16;
        case at::kHalf: return FMOE_F16;
        default: C10_THROW_ERROR(TypeError, c10::str("unsupported dtype ", t, "; expected float32, bfloat16 or float16"));
    }
}

void check(int status, const char* what) {
    if (status == FMOE_OK) return;
    if (status < 0) C10_THROW_ERROR(ValueError, c10::str(what, ": ", fmoe_last_error()));
    TORCH_CHECK(false, what, ": HIP error ", status, ": ", fmoe_last_error());
}

// every tensor lives on one HIP device
void require_gpu(std::initializer_list<const Tensor*> tensors) {
    const Tensor* first = nullptr;
    for (const Tensor* t : tensors) {
        if (!t->defined()) continue;
        TORCH_CHECK(t->is_cuda(), "flash_moe HIP ops need tensors on a ROCm GPU (got a CPU tensor); there is no CPU path");
        if (first == nullptr) first = t;
        else TORCH_CHECK(t->device() == first->device(), "tensors on different devices: ", first->device(), " and ", t->device());
    }
}

// sets the device of a call and tells its stream
struct Launch {
    explicit Launch(const Tensor& t) : guard(t.device()), stream(c10::hip::getCurrentHIPStream(t.device().index()).stream()) {}
    c10::DeviceGuard guard;
    hipStream_t stream;
};

Tensor workspace(const Tensor& like, size_t bytes) {
    return at::empty({(int64_t)(bytes ? bytes : 1)}, like.options().dtype(at::kByte));
}

void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
Tensor value(const OptTensor& t) { return t.has_value() ? *t : Tensor(); }

bool records_gradient(std::initializer_list<const Tensor*> tensors) {
    if (!at::GradMode::is_enabled()) return false;
    for (const Tensor* t : tensors)
        if (t->defined() && t->requires_grad()) return true;
    return false;
}

// Forward-mode derivatives are not implemented.  An input that carries a tangent is refused, as torch refuses it for an autograd
// function without one, whether or not a node would be recorded: an output without a tangent reads as a zero derivative.
void refuse_tangents(std::initializer_list<const Tensor*> tensors) {
    if (!c10::AutogradState::get_tls_state().get_fw_grad_mode()) return;
    for (const Tensor* t : tensors)
        if (t->defined() && t->_fw_grad(/*level=*/0).defined())
            C10_THROW_ERROR(NotImplementedError, "forward-mode differentiation is not implemented for the flash_moe ops");
}

// ---- router -----------------------------------------------------------------------------------------------------------
std::tuple<Tensor, Tensor, OptTensor> router_topk(const Tensor& router_logits, int64_t nk, int64_t K, bool with_gates, bool norm) {
    TORCH_CHECK_VALUE(router_logits.size(2) == nk, "router_logits.size(-1)=", router_logits.size(2), " does not match num_expert_keys=", nk);
    require_gpu({&router_logits});
    const int code = dtype_code(router_logits.scalar_type());
    const Tensor lp = router_logits.contiguous();
    const int64_t T = lp.size(1);
    Launch call(lp);
    Tensor scores = at::empty({T, K}, lp.options());
    Tensor indices = at::empty({T, K}, lp.options().dtype(at::kLong));
    Tensor gates = with_gates ? at::empty({T, K}, lp.options()) : Tensor();
    check(fmoe_router_topk(ptr(lp), T, (int)nk, (int)K, code, ptr(scores), (int64_t*)ptr(indices), ptr(gates), norm, call.stream), "flash_router");
    return {scores, indices, with_gates ? OptTensor(gates) : std::nullopt};
}

Tensor router_topk_backward(const Tensor& dscores, const Tensor& indices, int64_t nk) {
    TORCH_CHECK_VALUE(dscores.dim() == 2 && indices.sizes() == dscores.sizes() && indices.scalar_type() == at::kLong,
                      "expected dscores [T, K] and int64 indices of the same shape");
    require_gpu({&dscores, &indices});
    const int code = dtype_code(dscores.scalar_type());
    const Tensor ds = dscores.contiguous(), idx = indices.contiguous();
    Launch call(ds);
    Tensor out = at::empty({2, ds.size(0), nk}, ds.options());
    check(fmoe_router_topk_backward(ptr(ds), (const int64_t*)ptr(idx), ds.size(0), (int)nk, (int)ds.size(1), code, ptr(out), call.stream), "flash_router backward");
    return out;
}

struct RouterNode : torch::autograd::Function<RouterNode> {
    static variable_list forward(AutogradContext* ctx, const Tensor& router_logits, int64_t nk, int64_t K) {
        auto [scores, indices, gates] = router_topk(router_logits, nk, K, false, false);
        ctx->mark_non_differentiable({indices});
        ctx->set_materialize_grads(false);
        ctx->save_for_backward({indices});
        ctx->saved_data["nk"] = nk;
        return {scores, indices};
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        if (!grads[0].defined()) return {Tensor(), Tensor(), Tensor()};
        return {router_topk_backward(grads[0], ctx->get_saved_variables()[0], ctx->saved_data["nk"].toInt()), Tensor(), Tensor()};
    }
};

std::tuple<Tensor, Tensor> router_func(const Tensor& router_logits, int64_t nk, int64_t K) {
    refuse_tangents({&router_logits});
    if (records_gradient({&router_logits})) {
        auto out = RouterNode::apply(router_logits, nk, K);
        return {out[0], out[1]};
    }
    auto [scores, indices, gates] = router_topk(router_logits, nk, K, false, false);
    return {scores, indices};
}

// batch-norm state of a call: buffers (any of the three float types), mode and constants
struct Norm {
    Tensor mean, var, batches;
    bool training;
    double momentum, eps;
};

std::vector<Tensor> router_forward(const Tensor& tokens, const Tensor& gate_weight, const Tensor& mean, const Tensor& var,
                                   const OptTensor& batches, bool training, double momentum, double eps, int64_t nk, int64_t K,
                                   bool norm, bool split_query) {
    require_gpu({&tokens, &gate_weight, &mean, &var});
    const int code = dtype_code(tokens.scalar_type());
    const Tensor x = tokens.contiguous(), w = gate_weight.contiguous();
    const int64_t T = x.size(0), H = x.size(1);
    Launch call(x);
    Tensor logits = at::empty({T, 2 * nk}, x.options()), logits32 = at::empty({T, 2 * nk}, x.options().dtype(at::kFloat));
    Tensor scores = at::empty({T, K}, logits32.options()), indices = at::empty({T, K}, x.options().dtype(at::kLong));
    Tensor gates = at::empty({T, K}, x.options());
    const size_t bytes = fmoe_router_workspace_bytes(T, (int)H, (int)nk);
    Tensor ws = workspace(x, bytes);
    check((split_query ? fmoe_router_forward_split : fmoe_router_forward)(
              ptr(x), ptr(w), ptr(mean), ptr(var), (int64_t*)ptr(value(batches)), dtype_code(mean.scalar_type()), training,
              (float)momentum, (float)eps, T, (int)H, (int)nk, (int)K, code, norm, ptr(logits), (float*)ptr(logits32),
              (float*)ptr(scores), (int64_t*)ptr(indices), ptr(gates), ptr(ws), bytes, call.stream), "flash_router");
    Tensor stats;
    if (T > 0) {
        const int64_t at = (int64_t)fmoe_router_workspace_stats_offset(T, (int)H, (int)nk);
        stats = ws.slice(0, at, at + 2 * H * 4).view(at::kFloat);
    } else {
        stats = at::zeros({2 * H}, logits32.options());
    }
    return {logits, scores, indices, gates, logits32, stats};
}

Tensor route_backward(const Tensor& dgates, const Tensor& indices, const Tensor& logits32, int64_t nk, bool norm, const OptTensor& dlogits) {
    TORCH_CHECK_VALUE(dgates.dim() == 2 && indices.sizes() == dgates.sizes() && indices.scalar_type() == at::kLong,
                      "expected dgates [T, K] and int64 indices of the same shape");
    const int64_t T = dgates.size(0), K = dgates.size(1);
    TORCH_CHECK_VALUE(logits32.dim() == 2 && logits32.size(0) == T && logits32.size(1) == 2 * nk && logits32.scalar_type() == at::kFloat,
                      "expected fp32 logits of shape [T, 2*num_expert_keys]");
    const Tensor extra_in = value(dlogits);
    TORCH_CHECK_VALUE(!extra_in.defined() || (extra_in.sizes() == logits32.sizes() && extra_in.scalar_type() == dgates.scalar_type()),
                      "dlogits must have the shape of the logits and the dtype of dgates");
    require_gpu({&dgates, &indices, &logits32, &extra_in});
    const int code = dtype_code(dgates.scalar_type());
    const Tensor dg = dgates.contiguous(), idx = indices.contiguous(), lg = logits32.contiguous();
    const Tensor extra = extra_in.defined() ? extra_in.contiguous() : extra_in;
    Launch call(dg);
    Tensor out = at::empty_like(lg);
    check(fmoe_route_backward(ptr(dg), (const int64_t*)ptr(idx), (const float*)ptr(lg), ptr(extra), T, (int)nk, (int)K, code, norm,
                              (float*)ptr(out), call.stream), "route backward");
    return out;
}

std::tuple<Tensor, Tensor> router_prologue_backward(const Tensor& dlogits32, const Tensor& tokens, const Tensor& gate_weight,
                                                    const Tensor& stats, bool training) {
    const Tensor x = tokens.contiguous(), w = gate_weight.contiguous(), grad = dlogits32.contiguous();
    const int64_t T = x.size(0), H = x.size(1), nk = w.size(0) / 2;
    TORCH_CHECK_VALUE(grad.dim() == 2 && grad.size(0) == T && grad.size(1) == 2 * nk && grad.scalar_type() == at::kFloat,
                      "expected an fp32 gradient of shape [T, 2*num_expert_keys]");
    require_gpu({&x, &w, &grad, &stats});
    const int code = dtype_code(x.scalar_type());
    Launch call(x);
    Tensor dx = at::empty_like(x), dw = at::empty_like(w);
    const size_t bytes = fmoe_router_prologue_backward_workspace_bytes(T, (int)H, (int)nk, code);
    Tensor ws = workspace(x, bytes);
    check(fmoe_router_prologue_backward((const float*)ptr(grad), ptr(x), ptr(w), (const float*)ptr(stats), training, T, (int)H,
                                        (int)nk, code, ptr(dx), ptr(dw), ptr(ws), bytes, call.stream), "router prologue backward");
    return {dx, dw};
}

// Batch norm + gate product with gradients: (fp32 logits, logits in the activation dtype)
struct PrologueNode : torch::autograd::Function<PrologueNode> {
    static variable_list forward(AutogradContext* ctx, const Tensor& tokens, const Tensor& gate_weight, const Norm* norm) {
        const int64_t nk = gate_weight.size(0) / 2;
        auto out = router_forward(tokens, gate_weight, norm->mean, norm->var, norm->batches, norm->training, norm->momentum, norm->eps, nk, 0, false, false);
        ctx->set_materialize_grads(false);
        ctx->save_for_backward({tokens, gate_weight, out[5].clone()});
        ctx->saved_data["training"] = norm->training;
        return {out[4], out[0]};
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        Tensor grad;
        for (const Tensor& g : grads)
            if (g.defined()) grad = grad.defined() ? grad + g.to(at::kFloat) : g.to(at::kFloat);
        if (!grad.defined()) return {Tensor(), Tensor(), Tensor()};
        const auto saved = ctx->get_saved_variables();
        auto [dx, dw] = router_prologue_backward(grad, saved[0], saved[1], saved[2], ctx->saved_data["training"].toBool());
        return {dx, dw, Tensor()};
    }
};

std::tuple<Tensor, Tensor> router_prologue(const Tensor& tokens, const Tensor& gate_weight, const Tensor& mean, const Tensor& var,
                                           const OptTensor& batches, bool training, double momentum, double eps) {
    refuse_tangents({&tokens, &gate_weight});
    const Norm norm{mean, var, value(batches), training, momentum, eps};
    auto out = PrologueNode::apply(tokens, gate_weight, &norm);
    return {out[0], out[1]};
}

// ---- routed experts, PEER, PKM -------------------------------------------------------------------------------------------
// saved: where to put what a backward pass wants kept (undefined where the schedule keeps nothing), or NULL
Tensor expert_forward_impl(const Tensor& hidden_states, const Tensor& down, const Tensor& up, const Tensor& indices, const Tensor& weights,
                           int64_t algo, Tensor* saved) {
    TORCH_CHECK_VALUE(hidden_states.dim() == 2 && down.dim() == 2 && up.dim() == 2, "hidden_states, down_weights and up_weights must be 2-D");
    TORCH_CHECK_VALUE(indices.dim() == 2 && weights.sizes() == indices.sizes(), "indices and routing_weights must both be (num_tokens, num_experts_per_tok)");
    const int64_t T = hidden_states.size(0), H = hidden_states.size(1), E = down.size(0), K = indices.size(1);
    TORCH_CHECK_VALUE(down.size(1) == H && up.size(0) == E && up.size(1) == H, "down_weights and up_weights must be (num_experts, hidden_size)");
    TORCH_CHECK_VALUE(indices.size(0) == T, "indices has a different number of tokens than hidden_states");
    TORCH_CHECK_TYPE(indices.scalar_type() == at::kLong, "indices must be int64 (got ", indices.scalar_type(), ")");
    for (const Tensor* t : {&down, &up, &weights})
        TORCH_CHECK_TYPE(t->scalar_type() == hidden_states.scalar_type(), "down_weights, up_weights and routing_weights must have the dtype of hidden_states (",
                         hidden_states.scalar_type(), "), got ", t->scalar_type());
    require_gpu({&hidden_states, &down, &up, &indices, &weights});
    const int code = dtype_code(hidden_states.scalar_type());
    const Tensor x = hidden_states.contiguous(), wd = down.contiguous(), wu = up.contiguous(), idx = indices.contiguous(), g = weights.contiguous();
    Launch call(x);
    Tensor out = at::empty_like(x);
    const size_t bytes = saved != nullptr ? fmoe_expert_workspace_bytes(T, (int)H, E, (int)K, code)
                                          : fmoe_expert_workspace_bytes_algo(T, (int)H, E, (int)K, code, (int)algo);
    Tensor ws = bytes ? workspace(x, bytes) : Tensor();
    if (saved != nullptr) {
        const size_t kept = fmoe_expert_saved_bytes(T, (int)H, E, (int)K, code);
        if (kept) *saved = workspace(x, kept);
        check(fmoe_expert_forward_save(ptr(x), ptr(wd), ptr(wu), (const int64_t*)ptr(idx), ptr(g), T, (int)H, E, (int)K, code, ptr(out),
                                       ptr(*saved), kept, ptr(ws), bytes, call.stream), "flash_expert");
        return out;
    }
    check(fmoe_expert_forward_algo(ptr(x), ptr(wd), ptr(wu), (const int64_t*)ptr(idx), ptr(g), T, (int)H, E, (int)K, code, ptr(out),
                                   ptr(ws), bytes, (int)algo, call.stream), "flash_expert");
    return out;
}

Tensor expert_forward(const Tensor& hidden_states, const Tensor& down, const Tensor& up, const Tensor& indices, const Tensor& weights, int64_t algo) {
    return expert_forward_impl(hidden_states, down, up, indices, weights, algo, nullptr);
}

std::tuple<Tensor, Tensor, Tensor, Tensor> expert_backward_impl(const Tensor& dout, const Tensor& hidden_states, const Tensor& down,
                                                                const Tensor& up, const Tensor& indices, const Tensor& weights,
                                                                const Tensor& saved) {
    require_gpu({&dout, &hidden_states, &down, &up, &indices, &weights});
    TORCH_CHECK_VALUE(dout.sizes() == hidden_states.sizes() && dout.scalar_type() == hidden_states.scalar_type(),
                      "the output gradient must have the shape and dtype of hidden_states");
    const int code = dtype_code(hidden_states.scalar_type());
    const Tensor d = dout.contiguous(), x = hidden_states.contiguous(), wd = down.contiguous(), wu = up.contiguous(), idx = indices.contiguous(), g = weights.contiguous();
    const int64_t T = x.size(0), H = x.size(1), E = wd.size(0), K = idx.size(1);
    Launch call(x);
    Tensor dx = at::empty_like(x), dwd = at::empty_like(wd), dwu = at::empty_like(wu), dg = at::empty_like(g);
    const size_t bytes = fmoe_expert_backward_workspace_bytes(T, (int)H, E, (int)K, code);
    Tensor ws = workspace(x, bytes);
    check(fmoe_expert_backward_saved(ptr(d), ptr(x), ptr(wd), ptr(wu), (const int64_t*)ptr(idx), ptr(g), ptr(saved), T, (int)H, E, (int)K,
                                     code, ptr(dx), ptr(dwd), ptr(dwu), ptr(dg), ptr(ws), bytes, call.stream), "flash_expert backward");
    return {dx, dwd, dwu, dg};
}

std::tuple<Tensor, Tensor, Tensor, Tensor> expert_backward(const Tensor& dout, const Tensor& hidden_states, const Tensor& down,
                                                           const Tensor& up, const Tensor& indices, const Tensor& weights) {
    return expert_backward_impl(dout, hidden_states, down, up, indices, weights, Tensor());
}

struct ExpertNode : torch::autograd::Function<ExpertNode> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& down, const Tensor& up, const Tensor& indices, const Tensor& weights) {
        Tensor saved;
        Tensor out = expert_forward_impl(x, down, up, indices, weights, FMOE_EXPERT_AUTO, &saved);
        ctx->save_for_backward({x, down, up, indices, weights, saved});
        return out;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const auto s = ctx->get_saved_variables();
        auto [dx, dwd, dwu, dg] = expert_backward_impl(grads[0], s[0], s[1], s[2], s[3], s[4], s[5]);
        return {dx, dwd, dwu, Tensor(), dg};
    }
};

Tensor expert_func(const Tensor& x, const Tensor& down, const Tensor& up, const Tensor& indices, const Tensor& weights) {
    refuse_tangents({&x, &down, &up, &weights});
    if (records_gradient({&x, &down, &up, &weights})) return ExpertNode::apply(x, down, up, indices, weights);
    return expert_forward(x, down, up, indices, weights, FMOE_EXPERT_AUTO);
}

std::tuple<Tensor, Tensor, Tensor, Tensor> expert_bucketing(const Tensor& indices, int64_t E) {
    TORCH_CHECK_VALUE(indices.dim() == 2 && indices.scalar_type() == at::kLong, "indices must be an int64 tensor (num_tokens, num_experts_per_tok)");
    require_gpu({&indices});
    const Tensor idx = indices.contiguous();
    const int64_t T = idx.size(0), K = idx.size(1);
    Launch call(idx);
    const auto i32 = idx.options().dtype(at::kInt);
    Tensor offsets = at::empty({E + 1}, i32), pairs = at::empty({T * K}, i32), tokens = at::empty({T * K}, i32), experts = at::empty({T * K}, i32);
    const size_t bytes = fmoe_expert_bucket_workspace_bytes(E);
    Tensor ws = workspace(idx, bytes);
    check(fmoe_expert_bucket((const int64_t*)ptr(idx), T, (int)K, E, (int32_t*)ptr(offsets), (int32_t*)ptr(pairs), (int32_t*)ptr(tokens),
                             (int32_t*)ptr(experts), ptr(ws), bytes, call.stream), "flash_expert bucketing");
    return {tokens, offsets, pairs, experts};
}

Tensor peer_forward(const Tensor& hidden_states, const Tensor& down, const Tensor& up, const Tensor& weights, const Tensor& indices) {
    TORCH_CHECK_VALUE(hidden_states.dim() == 2 && down.dim() == 2 && up.sizes() == down.sizes(), "expected hidden_states [T, H] and down_embed / up_embed [E, H]");
    TORCH_CHECK_VALUE(indices.dim() == 2 && weights.sizes() == indices.sizes() && indices.size(0) == hidden_states.size(0),
                      "indices and routing_weights must both be (num_tokens, topk)");
    TORCH_CHECK_TYPE(indices.scalar_type() == at::kLong, "indices must be int64 (got ", indices.scalar_type(), ")");
    for (const Tensor* t : {&down, &up, &weights})
        TORCH_CHECK_TYPE(t->scalar_type() == hidden_states.scalar_type(), "down_embed, up_embed and routing_weights must have the dtype of hidden_states (",
                         hidden_states.scalar_type(), ")");
    const int64_t T = hidden_states.size(0), H = hidden_states.size(1), E = down.size(0), K = indices.size(1);
    TORCH_CHECK_VALUE(down.size(1) == H, "down_embed / up_embed rows must have hidden_size elements");
    require_gpu({&hidden_states, &down, &up, &weights, &indices});
    const int code = dtype_code(hidden_states.scalar_type());
    const Tensor x = hidden_states.contiguous(), wd = down.contiguous(), wu = up.contiguous(), w = weights.contiguous(), idx = indices.contiguous();
    Launch call(x);
    Tensor out = at::empty_like(x);
    const size_t bytes = fmoe_expert_workspace_bytes_algo(T, (int)H, E, (int)K, code, FMOE_EXPERT_AUTO);
    Tensor ws = workspace(x, bytes);
    check(fmoe_peer_forward(ptr(x), ptr(wd), ptr(wu), ptr(w), (const int64_t*)ptr(idx), T, (int)H, E, (int)K, code, ptr(out), ptr(ws),
                            bytes, call.stream), "peer");
    return out;
}

Tensor pkm_forward(const Tensor& values, const Tensor& weights, const Tensor& indices) {
    TORCH_CHECK_VALUE(values.dim() == 2 && indices.dim() == 2 && weights.sizes() == indices.sizes(), "expected values [E, H] and routing_weights / indices [T, topk]");
    TORCH_CHECK_TYPE(indices.scalar_type() == at::kLong, "indices must be int64 (got ", indices.scalar_type(), ")");
    TORCH_CHECK_TYPE(weights.scalar_type() == values.scalar_type(), "routing_weights has dtype ", weights.scalar_type(), ", values has ", values.scalar_type());
    require_gpu({&values, &weights, &indices});
    const int code = dtype_code(values.scalar_type());
    const Tensor v = values.contiguous(), w = weights.contiguous(), idx = indices.contiguous();
    const int64_t E = v.size(0), H = v.size(1), T = idx.size(0), K = idx.size(1);
    Launch call(v);
    Tensor out = at::empty({T, H}, v.options());
    const size_t bytes = fmoe_pkm_workspace_bytes(T, (int)H, E, (int)K, code);
    Tensor ws = workspace(v, bytes);
    check(fmoe_pkm_forward(ptr(v), ptr(w), (const int64_t*)ptr(idx), T, (int)H, E, (int)K, code, ptr(out), ptr(ws), bytes, call.stream), "pkm");
    return out;
}

struct PeerNode : torch::autograd::Function<PeerNode> {
    static Tensor forward(AutogradContext*, const Tensor& x, const Tensor& down, const Tensor& up, const Tensor& weights, const Tensor& indices) {
        return peer_forward(x, down, up, weights, indices);
    }
    static variable_list backward(AutogradContext*, variable_list) {
        C10_THROW_ERROR(NotImplementedError, "PEER backward is not implemented (nor is it in the reference)");
    }
};
Tensor peer_func(const Tensor& x, const Tensor& down, const Tensor& up, const Tensor& weights, const Tensor& indices) {
    refuse_tangents({&x, &down, &up, &weights});
    if (records_gradient({&x, &down, &up, &weights})) return PeerNode::apply(x, down, up, weights, indices);
    return peer_forward(x, down, up, weights, indices);
}

struct PkmNode : torch::autograd::Function<PkmNode> {
    static Tensor forward(AutogradContext*, const Tensor& values, const Tensor& weights, const Tensor& indices) { return pkm_forward(values, weights, indices); }
    static variable_list backward(AutogradContext*, variable_list) {
        C10_THROW_ERROR(NotImplementedError, "PKM backward is not implemented (nor is it in the reference)");
    }
};
Tensor pkm_func(const Tensor& values, const Tensor& weights, const Tensor& indices) {
    refuse_tangents({&values, &weights});
    if (records_gradient({&values, &weights})) return PkmNode::apply(values, weights, indices);
    return pkm_forward(values, weights, indices);
}

// ---- shared MLP ------------------------------------------------------------------------------------------------------------
void check_mlp_weights(const Tensor& x, const Tensor& gate, const Tensor& up, const Tensor& down) {
    const int64_t H = x.size(-1), I = gate.size(0);
    TORCH_CHECK_VALUE(gate.dim() == 2 && up.dim() == 2 && down.dim() == 2 && gate.size(1) == H && up.size(0) == I && up.size(1) == H &&
                          down.size(0) == H && down.size(1) == I,
                      "expected gate_weight/up_weight (intermediate, hidden) and down_weight (hidden, intermediate)");
    for (const Tensor* t : {&gate, &up, &down})
        TORCH_CHECK_TYPE(t->scalar_type() == x.scalar_type(), "all weights must have the dtype of x (", x.scalar_type(), "), got ", t->scalar_type());
}

Tensor contiguous_residual(const Tensor& residual, const Tensor& x) {
    if (!residual.defined()) return residual;
    TORCH_CHECK_VALUE(residual.sizes() == x.sizes() && residual.scalar_type() == x.scalar_type(), "residual must have the shape and dtype of x");
    return residual.contiguous();
}

Tensor mlp_forward(const Tensor& x_in, const Tensor& gate, const Tensor& up, const Tensor& down, const OptTensor& residual) {
    check_mlp_weights(x_in, gate, up, down);
    const Tensor res_in = value(residual);
    require_gpu({&x_in, &gate, &up, &down, &res_in});
    const int code = dtype_code(x_in.scalar_type());
    const Tensor x = x_in.contiguous(), wg = gate.contiguous(), wu = up.contiguous(), wd = down.contiguous(), res = contiguous_residual(res_in, x_in);
    const int64_t H = x.size(-1), I = wg.size(0), T = H ? x.numel() / H : 0;
    Launch call(x);
    Tensor out = at::empty_like(x);
    const size_t bytes = fmoe_mlp_workspace_bytes(T, (int)H, (int)I, code);
    Tensor ws = workspace(x, bytes);
    check(fmoe_mlp_forward(ptr(x), ptr(wg), ptr(wu), ptr(wd), T, (int)H, (int)I, code, ptr(res), ptr(out), ptr(ws), bytes, call.stream), "flash_mlp");
    return out;
}

// out and a [2, T, I] buffer: the gate and up products
std::tuple<Tensor, Tensor> mlp_forward_saving(const Tensor& x_in, const Tensor& gate, const Tensor& up, const Tensor& down, const OptTensor& residual) {
    check_mlp_weights(x_in, gate, up, down);
    const Tensor res_in = value(residual);
    require_gpu({&x_in, &gate, &up, &down, &res_in});
    const int code = dtype_code(x_in.scalar_type());
    const Tensor x = x_in.contiguous(), wg = gate.contiguous(), wu = up.contiguous(), wd = down.contiguous(), res = contiguous_residual(res_in, x_in);
    const int64_t H = x.size(-1), I = wg.size(0), T = H ? x.numel() / H : 0;
    Launch call(x);
    Tensor saved = at::empty({2, T, I}, x.options()), act = at::empty({T, I}, x.options()), out = at::empty_like(x);
    const size_t bytes = fmoe_mlp_down_workspace_bytes(T, (int)H, (int)I, code);
    Tensor ws = bytes ? workspace(x, bytes) : Tensor();
    check(fmoe_mlp_gate_up_save(ptr(x), ptr(wg), ptr(wu), T, (int)H, (int)I, code, ptr(act), ptr(saved), call.stream), "flash_mlp");
    check(fmoe_mlp_down_ws(ptr(act), ptr(wd), T, (int)H, (int)I, code, ptr(res), ptr(out), ptr(ws), bytes, call.stream), "flash_mlp");
    return {out, saved};
}

std::tuple<Tensor, Tensor, Tensor, Tensor> mlp_backward(const Tensor& dout, const Tensor& x_in, const Tensor& gate, const Tensor& up,
                                                        const Tensor& down, const OptTensor& products) {
    const Tensor saved = value(products);
    require_gpu({&dout, &x_in, &gate, &up, &down});
    TORCH_CHECK_VALUE(dout.sizes() == x_in.sizes() && dout.scalar_type() == x_in.scalar_type(), "the output gradient must have the shape and dtype of x");
    const int code = dtype_code(x_in.scalar_type());
    const Tensor x = x_in.contiguous(), dy = dout.contiguous(), wg = gate.contiguous(), wu = up.contiguous(), wd = down.contiguous();
    const int64_t H = x.size(-1), I = wg.size(0), T = H ? x.numel() / H : 0;
    TORCH_CHECK_VALUE(!saved.defined() || (saved.dim() == 3 && saved.size(0) == 2 && saved.size(1) == T && saved.size(2) == I &&
                                           saved.scalar_type() == x.scalar_type() && saved.is_contiguous()),
                      "saved must be the contiguous [2, T, I] tensor mlp_forward_saving returned");
    Launch call(x);
    // the two [I, H] gradients sit behind each other in one buffer: the library then forms them as one [2I, H] product
    Tensor dwgu = at::empty({2 * I, H}, wg.options());
    Tensor dwg = dwgu.narrow(0, 0, I), dwu = dwgu.narrow(0, I, I), dx = at::empty_like(x), dwd = at::empty_like(wd);
    if (T == 0) return {dx, dwg.zero_(), dwu.zero_(), dwd.zero_()};
    const size_t bytes = saved.defined() ? fmoe_mlp_backward_saved_workspace_bytes(T, (int)H, (int)I, code)
                                         : fmoe_mlp_backward_workspace_bytes(T, (int)H, (int)I, code);
    Tensor ws = workspace(x, bytes);
    check(fmoe_mlp_backward(ptr(dy), ptr(x), ptr(wg), ptr(wu), ptr(wd), ptr(saved), T, (int)H, (int)I, code, ptr(dx), ptr(dwg), ptr(dwu),
                            ptr(dwd), ptr(ws), bytes, call.stream), "flash_mlp backward");
    return {dx, dwg, dwu, dwd};
}

struct MlpNode : torch::autograd::Function<MlpNode> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& gate, const Tensor& up, const Tensor& down) {
        if (x.numel() == 0) {
            // nothing to keep for an empty batch: the backward returns zero gradients of the right shapes
            ctx->save_for_backward({x, gate, up, down});
            return mlp_forward(x, gate, up, down, std::nullopt);
        }
        auto [out, saved] = mlp_forward_saving(x, gate, up, down, std::nullopt);
        ctx->save_for_backward({x, gate, up, down, saved});
        return out;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const auto s = ctx->get_saved_variables();
        auto [dx, dwg, dwu, dwd] = mlp_backward(grads[0], s[0], s[1], s[2], s[3], s.size() > 4 ? OptTensor(s[4]) : std::nullopt);
        return {dx, dwg, dwu, dwd};
    }
};

Tensor mlp_func(const Tensor& x, const Tensor& gate, const Tensor& up, const Tensor& down) {
    refuse_tangents({&x, &gate, &up, &down});
    if (records_gradient({&x, &gate, &up, &down})) return MlpNode::apply(x, gate, up, down);
    return mlp_forward(x, gate, up, down, std::nullopt);
}

std::tuple<Tensor, Tensor> swiglu_backward(const Tensor& a, const Tensor& b, const Tensor& dc) {
    TORCH_CHECK_VALUE(a.sizes() == b.sizes() && a.sizes() == dc.sizes() && a.scalar_type() == b.scalar_type() && a.scalar_type() == dc.scalar_type(),
                      "a, b and dc must have one shape and dtype");
    require_gpu({&a, &b, &dc});
    const int code = dtype_code(a.scalar_type());
    const Tensor ac = a.contiguous(), bc = b.contiguous(), dcc = dc.contiguous();
    const int64_t cols = ac.size(-1);
    Launch call(ac);
    Tensor da = at::empty_like(ac), db = at::empty_like(bc);
    check(fmoe_swiglu_backward(ptr(dcc), ptr(ac), ptr(bc), cols ? ac.numel() / cols : 0, (int)cols, code, ptr(da), ptr(db), call.stream), "swiglu backward");
    return {da, db};
}

// ---- the whole block ---------------------------------------------------------------------------------------------------------
struct BlockShape {
    int64_t T, H, I, E, nk, K;
    int code;
    bool norm;
};

BlockShape check_block(const Tensor& x, const Tensor& wg, const Tensor& wu, const Tensor& wd, const Tensor& wr, const Tensor& ed,
                       const Tensor& eu, const Norm& bn, int64_t nk, int64_t K, bool norm) {
    const int64_t H = x.size(-1), I = wg.size(0), E = ed.size(0), T = H ? x.numel() / H : 0;
    TORCH_CHECK_VALUE(wr.dim() == 2 && wr.size(0) == 2 * nk && wr.size(1) == H, "expected tokens [T, H] and a router gate weight [2*num_expert_keys, H]");
    TORCH_CHECK_VALUE(wg.dim() == 2 && wu.dim() == 2 && wd.dim() == 2 && wg.size(1) == H && wu.size(0) == I && wu.size(1) == H && wd.size(0) == H && wd.size(1) == I,
                      "expected gate/up projection weights [I, H] and a down projection weight [H, I]");
    TORCH_CHECK_VALUE(ed.dim() == 2 && eu.dim() == 2 && ed.size(1) == H && eu.size(0) == E && eu.size(1) == H, "expected expert tables [E, H]");
    TORCH_CHECK_VALUE(nk * nk <= E, "num_expert_keys**2 = ", nk * nk, " exceeds the ", E, " rows of the expert tables");
    for (const Tensor* w : {&wg, &wu, &wd, &wr, &ed, &eu})
        TORCH_CHECK_TYPE(w->scalar_type() == x.scalar_type(), "all weights must have the tokens' dtype ", x.scalar_type());
    TORCH_CHECK_VALUE(!(bn.training && T == 1), "Expected more than 1 value per channel when training, got input size (1, ", H, ")");
    TORCH_CHECK_VALUE(bn.mean.is_contiguous() && bn.var.is_contiguous() && bn.mean.scalar_type() == bn.var.scalar_type(),
                      "running statistics must be contiguous and of one dtype");
    require_gpu({&x, &wg, &wu, &wd, &wr, &ed, &eu, &bn.mean, &bn.var});
    return {T, H, I, E, nk, K, dtype_code(x.scalar_type()), norm};
}

// router logits in the layout the block returns them, [2, T, nk] with a token's two halves side by side in memory
Tensor empty_logits(const Tensor& x, int64_t T, int64_t nk) { return at::empty_strided({2, T, nk}, {nk, 2 * nk, 1}, x.options()); }

std::vector<Tensor> block_forward(const Tensor& hidden_states, const Tensor& gate, const Tensor& up, const Tensor& down,
                                  const Tensor& router_gate, const Tensor& down_embed, const Tensor& up_embed, const Norm& bn,
                                  int64_t nk, int64_t K, bool norm, bool return_routing) {
    const BlockShape b = check_block(hidden_states, gate, up, down, router_gate, down_embed, up_embed, bn, nk, K, norm);
    const Tensor x = hidden_states.contiguous(), wg = gate.contiguous(), wu = up.contiguous(), wd = down.contiguous(), wr = router_gate.contiguous(),
                 ed = down_embed.contiguous(), eu = up_embed.contiguous();
    Launch call(x);
    Tensor out = at::empty_like(x), logits = empty_logits(x, b.T, nk), indices, gates;
    if (return_routing) {
        indices = at::empty({b.T, K}, x.options().dtype(at::kLong));
        gates = at::empty({b.T, K}, x.options());
    }
    const size_t bytes = fmoe_block_workspace_bytes(b.T, (int)b.H, (int)b.I, (int)nk, b.E, (int)K, b.code);
    Tensor ws = workspace(x, bytes);
    check(fmoe_block_forward(ptr(x), ptr(wg), ptr(wu), ptr(wd), ptr(wr), ptr(ed), ptr(eu), ptr(bn.mean), ptr(bn.var), (int64_t*)ptr(bn.batches),
                             dtype_code(bn.mean.scalar_type()), bn.training, (float)bn.momentum, (float)bn.eps, b.T, (int)b.H, (int)b.I,
                             b.E, (int)nk, (int)K, b.code, norm, ptr(out), ptr(logits), (int64_t*)ptr(indices), ptr(gates), ptr(ws), bytes,
                             call.stream), "flash_moe block");
    if (return_routing) return {out, logits, indices, gates};
    return {out, logits};
}

struct BlockNode : torch::autograd::Function<BlockNode> {
    static variable_list forward(AutogradContext* ctx, const Tensor& hidden_states, const Tensor& gate, const Tensor& up, const Tensor& down,
                                 const Tensor& router_gate, const Tensor& down_embed, const Tensor& up_embed, const Norm* bn, int64_t nk,
                                 int64_t K, bool norm) {
        const BlockShape b = check_block(hidden_states, gate, up, down, router_gate, down_embed, up_embed, *bn, nk, K, norm);
        const Tensor x = hidden_states.contiguous(), wg = gate.contiguous(), wu = up.contiguous(), wd = down.contiguous(),
                     wr = router_gate.contiguous(), ed = down_embed.contiguous(), eu = up_embed.contiguous();
        Launch call(x);
        Tensor out = at::empty_like(x), logits = empty_logits(x, b.T, nk);
        const size_t bytes = fmoe_block_workspace_bytes(b.T, (int)b.H, (int)b.I, (int)nk, b.E, (int)K, b.code);
        const size_t saved_bytes = fmoe_block_saved_bytes(b.T, (int)b.H, (int)b.I, (int)nk, b.E, (int)K, b.code);
        Tensor ws = workspace(x, bytes), saved = workspace(x, saved_bytes);
        check(fmoe_block_forward_save(ptr(x), ptr(wg), ptr(wu), ptr(wd), ptr(wr), ptr(ed), ptr(eu), ptr(bn->mean), ptr(bn->var),
                                      (int64_t*)ptr(bn->batches), dtype_code(bn->mean.scalar_type()), bn->training, (float)bn->momentum,
                                      (float)bn->eps, b.T, (int)b.H, (int)b.I, b.E, (int)nk, (int)K, b.code, norm, ptr(out), ptr(logits),
                                      ptr(saved), saved_bytes, ptr(ws), bytes, call.stream), "flash_moe block");
        ctx->set_materialize_grads(false);
        ctx->save_for_backward({x, wg, wu, wd, wr, ed, eu, saved});
        ctx->saved_data["training"] = bn->training;
        ctx->saved_data["K"] = K;
        ctx->saved_data["norm"] = norm;
        return {out, logits};
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        variable_list none(11);
        if (!grads[0].defined() && !grads[1].defined()) return none;
        const auto s = ctx->get_saved_variables();
        const Tensor &x = s[0], &wg = s[1], &wu = s[2], &wd = s[3], &wr = s[4], &ed = s[5], &eu = s[6], &saved = s[7];
        const int64_t H = x.size(-1), T = x.numel() / H, I = wg.size(0), E = ed.size(0), nk = wr.size(0) / 2, K = ctx->saved_data["K"].toInt();
        const int code = dtype_code(x.scalar_type());
        Launch call(x);
        const Tensor dout = grads[0].defined() ? grads[0].contiguous() : at::zeros_like(x);
        const Tensor dlogits = grads[1].defined() ? grads[1].contiguous() : Tensor();
        Tensor dwgu = at::empty({2 * I, H}, wg.options());      // one buffer: the library forms both gradients as one product
        Tensor dwg = dwgu.narrow(0, 0, I), dwu = dwgu.narrow(0, I, I);
        Tensor dx = at::empty_like(x), dwd = at::empty_like(wd), dwr = at::empty_like(wr), ded = at::empty_like(ed), deu = at::empty_like(eu);
        const size_t bytes = fmoe_block_backward_workspace_bytes(T, (int)H, (int)I, (int)nk, E, (int)K, code);
        Tensor ws = workspace(x, bytes);
        check(fmoe_block_backward(ptr(dout), ptr(dlogits), ptr(x), ptr(wg), ptr(wu), ptr(wd), ptr(wr), ptr(ed), ptr(eu), ptr(saved),
                                  ctx->saved_data["training"].toBool(), T, (int)H, (int)I, E, (int)nk, (int)K, code,
                                  ctx->saved_data["norm"].toBool(), ptr(dx), ptr(dwg), ptr(dwu), ptr(dwd), ptr(dwr), ptr(ded), ptr(deu),
                                  ptr(ws), bytes, call.stream), "flash_moe block backward");
        none[0] = dx; none[1] = dwg; none[2] = dwu; none[3] = dwd; none[4] = dwr; none[5] = ded; none[6] = deu;
        return none;
    }
};

std::vector<Tensor> block(const Tensor& hidden_states, const Tensor& gate, const Tensor& up, const Tensor& down, const Tensor& router_gate,
                          const Tensor& down_embed, const Tensor& up_embed, const Tensor& mean, const Tensor& var, const OptTensor& batches,
                          bool training, double momentum, double eps, int64_t nk, int64_t K, bool norm, bool differentiable, bool return_routing) {
    refuse_tangents({&hidden_states, &gate, &up, &down, &router_gate, &down_embed, &up_embed});
    const Norm bn{mean, var, value(batches), training, momentum, eps};
    if (differentiable && records_gradient({&hidden_states, &gate, &up, &down, &router_gate, &down_embed, &up_embed}))
        return BlockNode::apply(hidden_states, gate, up, down, router_gate, down_embed, up_embed, &bn, nk, K, norm);
    return block_forward(hidden_states, gate, up, down, router_gate, down_embed, up_embed, bn, nk, K, norm, return_routing);
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
#define FMOE_DEF(name) m.def(#name, torch::wrap_pybind_function(name))
    FMOE_DEF(router_topk);
    FMOE_DEF(router_topk_backward);
    FMOE_DEF(router_func);
    FMOE_DEF(router_forward);
    FMOE_DEF(route_backward);
    FMOE_DEF(router_prologue);
    FMOE_DEF(router_prologue_backward);
    FMOE_DEF(expert_forward);
    FMOE_DEF(expert_backward);
    FMOE_DEF(expert_func);
    FMOE_DEF(expert_bucketing);
    FMOE_DEF(peer_forward);
    FMOE_DEF(peer_func);
    FMOE_DEF(pkm_forward);
    FMOE_DEF(pkm_func);
    FMOE_DEF(mlp_forward);
    FMOE_DEF(mlp_forward_saving);
    FMOE_DEF(mlp_backward);
    FMOE_DEF(mlp_func);
    FMOE_DEF(swiglu_backward);
    FMOE_DEF(block);
#undef FMOE_DEF
}
