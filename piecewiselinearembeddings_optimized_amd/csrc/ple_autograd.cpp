// Autograd formulas of the PLE operators, in C++ so that a small training
// step's time is not spent in Python (nor in waiting for the interpreter
// between the caller's thread and the engine's): 256 x 8, 48 bins, d = 24,
// module forward and backward 132 -> 82 us a step against the same formulas
// registered from Python; recording the forward 37.7 -> 9.9 us.  What is left
// is the engine's own hand-over between threads (a multiplication and its
// backward: 47 us) and the module's Python.
//
// `forward`: the same contract as the reference
// (src/rtdl_num_embeddings_cuda/_autograd.py:9-96): the saved bin indices are
// non-differentiable, grads are not materialised, and the backward operator
// returns gradients for `x` and `weight` only.  (Integer outputs, as the
// indices and the ReLU pass bits are, are non-differentiable by their type;
// compiled autograd refuses nodes that mark outputs so themselves.)
//
// `forward_with_bias`: additionally returns the bias gradient from the same
// backward launch; `quant_dtype` is forwarded so the backward rounds the
// gradient, the fraction and the weights like the forward did.
//
// `forward_epilogue`: gradients for `x`, `weight`, `bias`, `lin_weight` and
// `lin_bias` from one backward launch, which reads the forward's ReLU pass
// bits (saved, non-differentiable).
//
// `encode`: the gradient of `x` from `encode_backward`.
//
// The operators are called through the dispatcher on both ways, so fake
// tensors, tracing and batched gradients see them, and the backwards have no
// state or side effects, so compiled autograd traces them into its graph
// (is_traceable) instead of breaking it for a call in eager mode.  Double backward and
// forward-mode derivatives are not implemented (as in the reference).

#include <ATen/ATen.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/library.h>

#include <tuple>

namespace {

using at::Tensor;
using c10::DispatchKeySet;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;
using OptTensor = c10::optional<Tensor>;
using Tensors2 = std::tuple<Tensor, Tensor>;
using Tensors3 = std::tuple<Tensor, Tensor, Tensor>;
using Tensors5 = std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor>;

template <typename Sig>
c10::TypedOperatorHandle<Sig> find_op(const char *name) {
    return c10::Dispatcher::singleton().findSchemaOrThrow(name, "").typed<Sig>();
}

#define PLE_OP(fn, name, ...)                                                                   \
    const c10::TypedOperatorHandle<__VA_ARGS__> &fn() {                                         \
        static const auto op = find_op<__VA_ARGS__>("rtdl_num_embeddings_cuda::" name);         \
        return op;                                                                              \
    }

PLE_OP(op_forward, "forward",
       Tensors2(const Tensor &, const Tensor &, const Tensor &, const Tensor &, const Tensor &, at::ScalarType))
PLE_OP(op_backward, "backward",
       Tensors2(const Tensor &, const Tensor &, const Tensor &, const Tensor &, const Tensor &, const Tensor &,
                const Tensor &, bool, bool))
PLE_OP(op_forward_with_bias, "forward_with_bias",
       Tensors2(const Tensor &, const Tensor &, const Tensor &, const Tensor &, const Tensor &, const Tensor &,
                at::ScalarType))
PLE_OP(op_backward_with_bias, "backward_with_bias",
       Tensors3(const Tensor &, const Tensor &, const Tensor &, const Tensor &, const Tensor &, const Tensor &,
                const Tensor &, at::ScalarType, bool, bool, bool))
PLE_OP(op_forward_epilogue, "forward_epilogue",
       Tensors3(const Tensor &, const Tensor &, const Tensor &, const Tensor &, const Tensor &, const OptTensor &,
                const OptTensor &, const OptTensor &, bool, bool, at::ScalarType))
PLE_OP(op_backward_epilogue, "backward_epilogue",
       Tensors5(const Tensor &, const Tensor &, const Tensor &, const Tensor &, const Tensor &, const Tensor &,
                const Tensor &, const Tensor &, const OptTensor &, bool, at::ScalarType, bool, bool, bool, bool, bool))
PLE_OP(op_encode, "encode",
       Tensor(const Tensor &, const Tensor &, const Tensor &, const Tensor &, const Tensor &, int64_t))
PLE_OP(op_encode_backward, "encode_backward",
       Tensor(const Tensor &, const Tensor &, const Tensor &, const Tensor &, const Tensor &, const Tensor &))
#undef PLE_OP

bool wants(const Tensor &t) { return t.defined() && t.requires_grad(); }
bool wants(const OptTensor &t) { return t.has_value() && wants(*t); }

bool has_tangent(const Tensor &t) { return t.defined() && t._fw_grad(/*level=*/0).defined(); }
bool has_tangent(const OptTensor &t) { return t.has_value() && has_tangent(*t); }

// whether the call is recorded: grad mode, and an input that requires grad
template <typename... T>
bool recorded(const T &...t) {
    if (!at::GradMode::is_enabled() || !(wants(t) || ...)) return false;
    TORCH_CHECK_NOT_IMPLEMENTED(!(has_tangent(t) || ...), "The PLE operators have no forward-mode derivative.");
    return true;
}

DispatchKeySet below(DispatchKeySet ks) { return ks & c10::after_autograd_keyset; }

// bit i: gradient i is wanted
template <typename... T>
int64_t need_bits(const T &...t) {
    int64_t bits = 0, i = 0;
    ((bits |= static_cast<int64_t>(wants(t)) << i++), ...);
    return bits;
}

Tensor if_bit(int64_t bits, int i, Tensor t) { return (bits >> i) & 1 ? std::move(t) : Tensor(); }

struct Forward : torch::autograd::Function<Forward> {
    static constexpr bool is_traceable = true;
    static variable_list forward(AutogradContext *ctx, DispatchKeySet ks, const Tensor &x, const Tensor &edges,
                                 const Tensor &iw, const Tensor &nbins, const Tensor &weight,
                                 at::ScalarType output_dtype) {
        at::AutoDispatchBelowAutograd guard;
        auto [out, idx] = op_forward().redispatch(below(ks), x, edges, iw, nbins, weight, output_dtype);
        ctx->save_for_backward({x, edges, iw, nbins, weight, idx});
        ctx->saved_data["need"] = need_bits(x, weight);
        ctx->set_materialize_grads(false);
        return {out, idx};
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        variable_list r(7);
        if (!grads[0].defined()) return r;
        const auto s = ctx->get_saved_variables();
        const int64_t need = ctx->saved_data["need"].toInt();
        auto [gx, gw] = op_backward().call(grads[0].contiguous(), s[0], s[1], s[2], s[3], s[4], s[5], need & 1,
                                           (need >> 1) & 1);
        r[1] = if_bit(need, 0, gx);
        r[5] = if_bit(need, 1, gw);
        return r;
    }
};

Tensors2 forward(DispatchKeySet ks, const Tensor &x, const Tensor &edges, const Tensor &iw, const Tensor &nbins,
                 const Tensor &weight, at::ScalarType output_dtype) {
    if (!recorded(x, edges, iw, nbins, weight)) {
        at::AutoDispatchBelowAutograd guard;
        return op_forward().redispatch(below(ks), x, edges, iw, nbins, weight, output_dtype);
    }
    auto r = Forward::apply(ks, x, edges, iw, nbins, weight, output_dtype);
    return {r[0], r[1]};
}

struct ForwardWithBias : torch::autograd::Function<ForwardWithBias> {
    static constexpr bool is_traceable = true;
    static variable_list forward(AutogradContext *ctx, DispatchKeySet ks, const Tensor &x, const Tensor &edges,
                                 const Tensor &iw, const Tensor &nbins, const Tensor &weight, const Tensor &bias,
                                 at::ScalarType quant_dtype) {
        at::AutoDispatchBelowAutograd guard;
        auto [out, idx] = op_forward_with_bias().redispatch(below(ks), x, edges, iw, nbins, weight, bias, quant_dtype);
        ctx->save_for_backward({x, edges, iw, nbins, weight, idx});
        ctx->saved_data["need"] = need_bits(x, weight, bias);
        ctx->saved_data["quant"] = static_cast<int64_t>(quant_dtype);
        ctx->set_materialize_grads(false);
        return {out, idx};
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        variable_list r(8);
        if (!grads[0].defined()) return r;
        const auto s = ctx->get_saved_variables();
        const int64_t need = ctx->saved_data["need"].toInt();
        const auto quant = static_cast<at::ScalarType>(ctx->saved_data["quant"].toInt());
        auto [gx, gw, gb] = op_backward_with_bias().call(grads[0].contiguous(), s[0], s[1], s[2], s[3], s[4], s[5],
                                                         quant, need & 1, (need >> 1) & 1, (need >> 2) & 1);
        r[1] = if_bit(need, 0, gx);
        r[5] = if_bit(need, 1, gw);
        r[6] = if_bit(need, 2, gb);
        return r;
    }
};

Tensors2 forward_with_bias(DispatchKeySet ks, const Tensor &x, const Tensor &edges, const Tensor &iw,
                           const Tensor &nbins, const Tensor &weight, const Tensor &bias, at::ScalarType quant_dtype) {
    if (!recorded(x, edges, iw, nbins, weight, bias)) {
        at::AutoDispatchBelowAutograd guard;
        return op_forward_with_bias().redispatch(below(ks), x, edges, iw, nbins, weight, bias, quant_dtype);
    }
    auto r = ForwardWithBias::apply(ks, x, edges, iw, nbins, weight, bias, quant_dtype);
    return {r[0], r[1]};
}

struct ForwardEpilogue : torch::autograd::Function<ForwardEpilogue> {
    static constexpr bool is_traceable = true;
    static variable_list forward(AutogradContext *ctx, DispatchKeySet ks, const Tensor &x, const Tensor &edges,
                                 const Tensor &iw, const Tensor &nbins, const Tensor &weight, const OptTensor &bias,
                                 const OptTensor &lin_weight, const OptTensor &lin_bias, bool relu, bool save_mask,
                                 at::ScalarType quant_dtype) {
        at::AutoDispatchBelowAutograd guard;
        auto [out, idx, mask] = op_forward_epilogue().redispatch(below(ks), x, edges, iw, nbins, weight, bias,
                                                                 lin_weight, lin_bias, relu, save_mask, quant_dtype);
        ctx->save_for_backward({x, edges, iw, nbins, weight, idx, mask, lin_weight.value_or(Tensor())});
        ctx->saved_data["need"] = need_bits(x, weight, bias, lin_weight, lin_bias);
        ctx->saved_data["quant"] = static_cast<int64_t>(quant_dtype);
        ctx->saved_data["relu"] = relu;
        // (the flag, not the mask's size: an empty batch saves an empty mask)
        ctx->saved_data["save_mask"] = save_mask;
        ctx->set_materialize_grads(false);
        return {out, idx, mask};
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        variable_list r(12);
        if (!grads[0].defined()) return r;
        const auto s = ctx->get_saved_variables();
        const int64_t need = ctx->saved_data["need"].toInt();
        const auto quant = static_cast<at::ScalarType>(ctx->saved_data["quant"].toInt());
        const bool relu = ctx->saved_data["relu"].toBool();
        TORCH_CHECK(!relu || ctx->saved_data["save_mask"].toBool(),
                    "forward_epilogue was called with save_mask=False; its ReLU cannot be differentiated");
        auto [gx, gw, gb, glw, glb] = op_backward_epilogue().call(
            grads[0].contiguous(), s[0], s[1], s[2], s[3], s[4], s[5], s[6],
            s[7].defined() ? OptTensor(s[7]) : OptTensor(), relu, quant, need & 1, (need >> 1) & 1, (need >> 2) & 1,
            (need >> 3) & 1, (need >> 4) & 1);
        r[1] = if_bit(need, 0, gx);
        r[5] = if_bit(need, 1, gw);
        r[6] = if_bit(need, 2, gb);
        r[7] = if_bit(need, 3, glw);
        r[8] = if_bit(need, 4, glb);
        return r;
    }
};

Tensors3 forward_epilogue(DispatchKeySet ks, const Tensor &x, const Tensor &edges, const Tensor &iw,
                          const Tensor &nbins, const Tensor &weight, const OptTensor &bias,
                          const OptTensor &lin_weight, const OptTensor &lin_bias, bool relu, bool save_mask,
                          at::ScalarType quant_dtype) {
    if (!recorded(x, edges, iw, nbins, weight, bias, lin_weight, lin_bias)) {
        at::AutoDispatchBelowAutograd guard;
        return op_forward_epilogue().redispatch(below(ks), x, edges, iw, nbins, weight, bias, lin_weight, lin_bias,
                                                relu, save_mask, quant_dtype);
    }
    auto r = ForwardEpilogue::apply(ks, x, edges, iw, nbins, weight, bias, lin_weight, lin_bias, relu, save_mask,
                                    quant_dtype);
    return {r[0], r[1], r[2]};
}

struct Encode : torch::autograd::Function<Encode> {
    static constexpr bool is_traceable = true;
    static Tensor forward(AutogradContext *ctx, DispatchKeySet ks, const Tensor &x, const Tensor &edges,
                          const Tensor &iw, const Tensor &nbins, const Tensor &offsets, int64_t total_bins) {
        at::AutoDispatchBelowAutograd guard;
        ctx->save_for_backward({x, edges, iw, nbins, offsets});
        ctx->saved_data["need"] = need_bits(x);
        ctx->set_materialize_grads(false);
        return op_encode().redispatch(below(ks), x, edges, iw, nbins, offsets, total_bins);
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        variable_list r(7);
        if (!grads[0].defined() || ctx->saved_data["need"].toInt() == 0) return r;
        const auto s = ctx->get_saved_variables();
        r[1] = op_encode_backward().call(grads[0].contiguous(), s[0], s[1], s[2], s[3], s[4]);
        return r;
    }
};

Tensor encode(DispatchKeySet ks, const Tensor &x, const Tensor &edges, const Tensor &iw, const Tensor &nbins,
              const Tensor &offsets, int64_t total_bins) {
    if (!recorded(x, edges, iw, nbins, offsets)) {
        at::AutoDispatchBelowAutograd guard;
        return op_encode().redispatch(below(ks), x, edges, iw, nbins, offsets, total_bins);
    }
    return Encode::apply(ks, x, edges, iw, nbins, offsets, total_bins);
}

}  // namespace

TORCH_LIBRARY_IMPL(rtdl_num_embeddings_cuda, Autograd, m) {
    m.impl("forward", TORCH_FN(forward));
    m.impl("forward_with_bias", TORCH_FN(forward_with_bias));
    m.impl("forward_epilogue", TORCH_FN(forward_epilogue));
    m.impl("encode", TORCH_FN(encode));
}
