// The host side of the small calls in C++: at the reference's batch sizes a training step or a packed evaluation is bound by
// what the host does per layer (argument checks, allocations, the autograd node, the call across the language border), not by
// its 4 to 9 us kernels.  Each entry takes what the Python function of the same job takes, launches the same C entry point of
// libdifflogic_hip.so on torch's current stream, and returns None where the arguments are not the plain case (another type,
// device, stride, an empty tensor): the caller then goes on in Python, which knows every case and raises the errors.
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/extension.h>

#include "difflogic_hip.h"

namespace {

using torch::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

void check(int status, const char *what) {
    if (status == DL_OK) return;
    std::string text = std::string(what) + ": " + dl_status_string(status);
    if (status == DL_ERR_LAUNCH) text += std::string(" (") + dl_last_hip_error() + ")";
    if (status == DL_ERR_NOT_DIVISIBLE || status == DL_ERR_BIT_COUNT) throw py::value_error(text);
    throw std::runtime_error(text);
}

void *stream_of(const Tensor &t) { return (void *) c10::hip::getCurrentHIPStream(t.get_device()).stream(); }

// dtype code of activations and weights side by side, or -1
int layer_code(at::ScalarType x, at::ScalarType w) {
    if (x == at::kFloat) return w == at::kFloat ? DL_F32 : -1;
    if (x == at::kHalf) return w == at::kHalf ? DL_F16 : w == at::kFloat ? DL_F16_W32 : -1;
    if (x == at::kDouble) return w == at::kDouble ? DL_F64 : w == at::kFloat ? DL_F64_W32 : -1;
    return -1;
}

bool plain(const Tensor &t, c10::DeviceIndex device) { return t.is_cuda() && t.get_device() == device && t.is_contiguous(); }

bool index_of(const Tensor &t, c10::DeviceIndex device, int64_t numel) {
    return t.scalar_type() == at::kLong && t.dim() == 1 && t.size(0) == numel && plain(t, device);
}

// LogicLayerLogitsFunction without a schedule: feature-major x [in, B] and gate logits -> y [out, B].
struct LayerFunction : torch::autograd::Function<LayerFunction> {
    static Tensor forward(AutogradContext *ctx, const Tensor &x, const Tensor &logits, const Tensor &a, const Tensor &b,
                          const Tensor &start, const Tensor &idx, double scale, int64_t code) {
        const int64_t out_dim = logits.size(0);
        Tensor w = logits.detach();
        Tensor y = at::empty({out_dim, x.size(1)}, x.options()), probs = at::empty_like(w);
        check(dl_logic_forward_logits(x.const_data_ptr(), a.const_data_ptr<int64_t>(), b.const_data_ptr<int64_t>(),
                                      w.const_data_ptr(), y.mutable_data_ptr(), probs.mutable_data_ptr(), x.size(0), out_dim,
                                      x.size(1), (int) code, stream_of(x)),
              "logic_layer_cuda_forward_logits");
        ctx->save_for_backward({x, a, b, probs, start, idx});
        ctx->saved_data["scale"] = scale;
        ctx->saved_data["code"] = code;
        return y;
    }

    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const variable_list saved = ctx->get_saved_variables();
        const Tensor &x = saved[0], &a = saved[1], &b = saved[2], &probs = saved[3], &start = saved[4], &idx = saved[5];
        const double scale = ctx->saved_data["scale"].toDouble();
        const int code = (int) ctx->saved_data["code"].toInt();
        const c10::DeviceGuard guard(x.device());
        const Tensor gy = grads[0].contiguous();
        TORCH_CHECK(gy.scalar_type() == x.scalar_type() && gy.dim() == 2 && gy.size(0) == probs.size(0) && gy.size(1) == x.size(1)
                        && gy.device() == x.device(),
                    "expected grad_y [out,B] of x's dtype and device");
        const bool want_x = ctx->needs_input_grad(0), want_w = ctx->needs_input_grad(1);
        const int64_t in_dim = x.size(0), out_dim = probs.size(0), batch = x.size(1);
        const int64_t *ap = a.const_data_ptr<int64_t>(), *bp = b.const_data_ptr<int64_t>();
        const int64_t *sp = start.const_data_ptr<int64_t>(), *ip = idx.const_data_ptr<int64_t>();
        Tensor gx = want_x ? at::empty_like(x) : Tensor(), gw = want_w ? at::empty_like(probs) : Tensor();
        if (want_x && want_w)
            check(dl_logic_backward_both(x.const_data_ptr(), ap, bp, probs.const_data_ptr(), gy.const_data_ptr(), 1, sp, ip,
                                         gw.mutable_data_ptr(), gx.mutable_data_ptr(), in_dim, out_dim, batch, 0, scale, code,
                                         stream_of(x)),
                  "logic_layer_cuda_backward_both");
        else if (want_x)
            check(dl_logic_backward_x(x.const_data_ptr(), ap, bp, probs.const_data_ptr(), gy.const_data_ptr(), sp, ip,
                                      gx.mutable_data_ptr(), in_dim, out_dim, batch, scale, code, stream_of(x)),
                  "logic_layer_cuda_backward_x");
        else if (want_w)
            check(dl_logic_backward_logits(x.const_data_ptr(), ap, bp, gy.const_data_ptr(), probs.const_data_ptr(),
                                           gw.mutable_data_ptr(), in_dim, out_dim, batch, code, stream_of(x)),
                  "logic_layer_cuda_backward_w");
        return {gx, gw, Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
    }
};

// A training layer on x [B, in] as LogicLayer.forward_cuda runs one that has no schedule: y [B, out], a view of [out, B].
c10::optional<Tensor> train_layer(const Tensor &x, const Tensor &weights, const Tensor &a, const Tensor &b, const Tensor &start,
                                  const Tensor &idx, double scale) {
    if (!x.is_cuda() || x.dim() != 2 || weights.dim() != 2 || weights.size(1) != 16) return c10::nullopt;
    const c10::DeviceIndex device = x.get_device();
    const int code = layer_code(x.scalar_type(), weights.scalar_type());
    const int64_t out_dim = weights.size(0), in_dim = x.size(1);
    if (code < 0 || x.size(0) == 0 || in_dim == 0 || out_dim == 0 || !plain(weights, device) || !index_of(a, device, out_dim)
        || !index_of(b, device, out_dim) || !index_of(start, device, in_dim + 1) || !index_of(idx, device, 2 * out_dim))
        return c10::nullopt;
    const c10::DeviceGuard guard(x.device());
    return LayerFunction::apply(x.transpose(0, 1).contiguous(), weights, a, b, start, idx, scale, (int64_t) code).transpose(0, 1);
}

// GroupSumCudaFunction: feature-major x [out, B] -> scores [B, k].
struct GroupSumFunction : torch::autograd::Function<GroupSumFunction> {
    static Tensor forward(AutogradContext *ctx, const Tensor &x, int64_t k, double tau, int64_t code) {
        const int64_t out_dim = x.size(0), batch = x.size(1);
        Tensor y = at::empty({batch, k}, x.options());
        const int64_t bytes = dl_group_sum_workspace_bytes(out_dim, batch, k, (int) code);
        Tensor ws = at::empty({std::max<int64_t>(1, bytes)}, x.options().dtype(at::kByte));
        check(dl_group_sum_forward(x.const_data_ptr(), y.mutable_data_ptr(), ws.mutable_data_ptr(), out_dim, batch, k, tau,
                                   (int) code, stream_of(x)),
              "group_sum_forward");
        ctx->saved_data["out_dim"] = out_dim;
        ctx->saved_data["tau"] = tau;
        ctx->saved_data["code"] = code;
        return y;
    }

    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const Tensor g = grads[0].contiguous();
        const c10::DeviceGuard guard(g.device());
        const int64_t out_dim = ctx->saved_data["out_dim"].toInt(), batch = g.size(0), k = g.size(1);
        const int code = layer_code(g.scalar_type(), g.scalar_type());
        TORCH_CHECK(code == ctx->saved_data["code"].toInt() && g.is_cuda(), "expected the gradient of GroupSum in its dtype");
        Tensor gx = at::empty({out_dim, batch}, g.options());
        check(dl_group_sum_backward(g.const_data_ptr(), gx.mutable_data_ptr(), out_dim, batch, k, ctx->saved_data["tau"].toDouble(),
                                    code, stream_of(g)),
              "group_sum_backward");
        return {gx, Tensor(), Tensor(), Tensor()};
    }
};

// GroupSum on the transposed view [B, out] that a layer returns.
c10::optional<Tensor> group_sum(const Tensor &x, int64_t k, double tau) {
    if (!x.is_cuda() || x.dim() != 2 || x.numel() == 0 || x.stride(0) != 1 || x.stride(1) != x.size(0) || k <= 0
        || x.size(1) % k != 0)
        return c10::nullopt;
    const int code = layer_code(x.scalar_type(), x.scalar_type());
    if (code < 0) return c10::nullopt;
    const Tensor xt = x.transpose(0, 1);
    if (!xt.is_contiguous()) return c10::nullopt;
    const c10::DeviceGuard guard(x.device());
    return GroupSumFunction::apply(xt, k, tau, (int64_t) code);
}

// difflogic_cuda.eval_weights: one packed layer from its weights, on rows int64 [in, W] (W even).
c10::optional<Tensor> eval_weights(const Tensor &x, const Tensor &a, const Tensor &b, const Tensor &w) {
    if (!x.is_cuda() || x.dim() != 2 || x.scalar_type() != at::kLong || x.size(1) % 2 || w.dim() != 2 || w.size(1) != 16)
        return c10::nullopt;
    const c10::DeviceIndex device = x.get_device();
    const int code = layer_code(w.scalar_type(), w.scalar_type());
    const int64_t out_dim = w.size(0);
    if (code < 0 || !plain(x, device) || !plain(w, device) || !index_of(a, device, out_dim) || !index_of(b, device, out_dim))
        return c10::nullopt;
    const c10::DeviceGuard guard(x.device());
    Tensor y = at::empty({out_dim, x.size(1)}, x.options());
    check(dl_logic_eval_weights(x.const_data_ptr(), a.const_data_ptr<int64_t>(), b.const_data_ptr<int64_t>(), w.const_data_ptr(),
                                code, y.mutable_data_ptr(), x.size(0), out_dim, x.size(1) * 8, stream_of(x)),
          "logic_eval_weights");
    return y;
}

// difflogic_cuda.gate_ids_folded: (ids, state_out) of a layer, both uint8 [out].
c10::optional<std::tuple<Tensor, Tensor>> gate_ids_folded(const Tensor &w, const Tensor &a, const Tensor &b,
                                                          const c10::optional<Tensor> &state) {
    if (!w.is_cuda() || w.dim() != 2 || w.size(1) != 16) return c10::nullopt;
    const c10::DeviceIndex device = w.get_device();
    const int code = layer_code(w.scalar_type(), w.scalar_type());
    const int64_t out_dim = w.size(0);
    if (code < 0 || !plain(w, device) || !index_of(a, device, out_dim) || !index_of(b, device, out_dim)) return c10::nullopt;
    if (state && (state->scalar_type() != at::kByte || state->dim() != 1 || !plain(*state, device))) return c10::nullopt;
    const c10::DeviceGuard guard(w.device());
    Tensor both = at::empty({2, out_dim}, w.options().dtype(at::kByte));
    uint8_t *ids = both.mutable_data_ptr<uint8_t>();
    check(dl_gate_ids_folded(w.const_data_ptr(), code, a.const_data_ptr<int64_t>(), b.const_data_ptr<int64_t>(),
                             state ? state->const_data_ptr<uint8_t>() : nullptr, ids, ids + out_dim, out_dim, stream_of(w)),
          "gate_ids_folded");
    return std::make_tuple(both.select(0, 0), both.select(0, 1));
}

// difflogic_cuda.tensor_packbits_batch_major_rows: bool [B, F] -> int64 [F, row_bytes / 8].
c10::optional<Tensor> pack_rows(const Tensor &x, int64_t row_bytes) {
    if (!x.is_cuda() || x.dim() != 2 || x.scalar_type() != at::kBool || !x.is_contiguous() || row_bytes % 8
        || row_bytes * 8 < x.size(0))
        return c10::nullopt;
    const c10::DeviceGuard guard(x.device());
    Tensor out = at::empty({x.size(1), row_bytes / 8}, x.options().dtype(at::kLong));
    check(dl_tensor_packbits_batch_major_rows((const uint8_t *) x.const_data_ptr(), out.mutable_data_ptr(), x.size(0), x.size(1),
                                              row_bytes, stream_of(x)),
          "tensor_packbits_batch_major_rows");
    return out;
}

// difflogic_cuda.groupbitsum of padded int64 rows: int32 [W * 64 - pad, k].
c10::optional<Tensor> count_rows(const Tensor &b, int64_t pad, int64_t k) {
    if (!b.is_cuda() || b.dim() != 2 || b.scalar_type() != at::kLong || !b.is_contiguous() || k <= 0 || b.size(0) % k || pad < 0
        || b.size(1) * 64 < pad)
        return c10::nullopt;
    const c10::DeviceGuard guard(b.device());
    Tensor out = at::empty({b.size(1) * 64 - pad, k}, b.options().dtype(at::kInt));
    check(dl_groupbitsum(b.const_data_ptr(), out.mutable_data_ptr<int32_t>(), b.size(0), b.size(1), 64, (int) pad, (int) k,
                         stream_of(b)),
          "groupbitsum");
    return out;
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    typedef py::call_guard<py::gil_scoped_release> unlocked;
    m.def("train_layer", &train_layer, unlocked());
    m.def("group_sum", &group_sum, unlocked());
    m.def("eval_weights", &eval_weights, unlocked());
    m.def("gate_ids_folded", &gate_ids_folded, unlocked());
    m.def("pack_rows", &pack_rows, unlocked());
    m.def("count_rows", &count_rows, unlocked());
}
