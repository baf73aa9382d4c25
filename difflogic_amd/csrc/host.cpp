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

// Saved tensors may have been through a caller's hooks: [x, a, b, probabilities, start, idx] for each layer, as they were saved
// (code(layer): the layer's dtype code then; the layers are a chain on one device).
template <typename Code>
void check_saved(const variable_list &saved, const Code &code) {
    for (size_t i = 0; i + 5 < saved.size(); i += 6) {
        const Tensor &x = saved[i], &probs = saved[i + 3];
        TORCH_CHECK(x.is_cuda() && x.dim() == 2 && probs.dim() == 2 && probs.size(1) == 16
                        && layer_code(x.scalar_type(), probs.scalar_type()) == code(i / 6),
                    "saved tensors have to come back as they were: in their shape and dtype");
        const c10::DeviceIndex device = saved[0].get_device();
        const int64_t in_dim = x.size(0), out_dim = probs.size(0);
        TORCH_CHECK(i == 0 || (in_dim == saved[i - 3].size(0) && x.size(1) == saved[0].size(1)),
                    "saved tensors have to come back as they were: in their shape and dtype");
        TORCH_CHECK(plain(x, device) && plain(probs, device) && index_of(saved[i + 1], device, out_dim)
                        && index_of(saved[i + 2], device, out_dim) && index_of(saved[i + 4], device, in_dim + 1)
                        && index_of(saved[i + 5], device, 2 * out_dim),
                    "saved tensors have to come back as they were: contiguous and on their device");
    }
}

// A layer's walk along its evaluation schedule: difflogic_cuda.EvalSchedule and the plan of its one-pass backward
// ([verts, neuron, flip, dst, fix_vertex, fix_start]; none: the layer has no schedule), whether the inputs at several
// positions are finished in the launch (DL_FIX_POSITIONS), and which of the kernels take the schedule.
struct Walk {
    std::vector<Tensor> tables;
    int64_t steps = 0, n_fix = 0, rows = 0;
    bool here = false, forward = false, weights = false;

    const int32_t *i32(int i) const { return tables[i].const_data_ptr<int32_t>(); }
    const uint8_t *flip() const { return tables[2].const_data_ptr<uint8_t>(); }
};

bool fits(const Walk &w, c10::DeviceIndex device) {
    if (w.tables.empty()) return true;
    if (w.tables.size() != 6 || w.steps < 0 || w.n_fix < 0 || w.rows < 0) return false;
    const int64_t sizes[6] = {w.steps + 1, w.steps, w.steps, w.steps + 1, w.n_fix, w.n_fix + 1 + w.rows};
    for (int i = 0; i < 6; ++i)
        if (w.tables[i].scalar_type() != (i == 2 ? at::kByte : at::kInt) || w.tables[i].numel() != sizes[i] || !plain(w.tables[i], device))
            return false;
    return true;
}

Tensor forward_into(const Tensor &x, const Tensor &a, const Tensor &b, const Tensor &logits, const Tensor &probs, int code,
                    const Walk &walk) {
    const int64_t out_dim = logits.size(0);
    Tensor y = at::empty({out_dim, x.size(1)}, x.options());
    int st = DL_ERR_TOO_LARGE;
    if (!walk.tables.empty() && walk.forward)
        st = dl_logic_forward_chained(x.const_data_ptr(), walk.i32(0), walk.i32(1), walk.flip(), walk.steps, logits.const_data_ptr(),
                                      y.mutable_data_ptr(), probs.mutable_data_ptr(), x.size(0), out_dim, x.size(1),
                                      code | DL_ROWS_ANY, stream_of(x));
    if (st == DL_ERR_TOO_LARGE)
        st = dl_logic_forward_logits(x.const_data_ptr(), a.const_data_ptr<int64_t>(), b.const_data_ptr<int64_t>(),
                                     logits.const_data_ptr(), y.mutable_data_ptr(), probs.mutable_data_ptr(), x.size(0), out_dim,
                                     x.size(1), code, stream_of(x));
    check(st, "logic_layer_cuda_forward_logits");
    return y;
}

void backward_both_into(const Tensor &x, const Tensor &a, const Tensor &b, const Tensor &probs, const Tensor &gy,
                        const Tensor &start, const Tensor &idx, const Tensor &gw, const Tensor &gx, int64_t gdiv_classes,
                        double scale, bool softmax, int code) {
    check(dl_logic_backward_both(x.const_data_ptr(), a.const_data_ptr<int64_t>(), b.const_data_ptr<int64_t>(),
                                 probs.const_data_ptr(), gy.const_data_ptr(), softmax ? 1 : 0, start.const_data_ptr<int64_t>(),
                                 idx.const_data_ptr<int64_t>(), gw.mutable_data_ptr(), gx.mutable_data_ptr(), x.size(0),
                                 probs.size(0), x.size(1), gdiv_classes, scale, code, stream_of(x)),
          "logic_layer_cuda_backward_both");
}

// LogicLayerLogitsFunction: feature-major x [in, B] and gate logits -> y [out, B].
struct LayerFunction : torch::autograd::Function<LayerFunction> {
    static Tensor forward(AutogradContext *ctx, const Tensor &x, const Tensor &logits, const Tensor &a, const Tensor &b,
                          const Tensor &start, const Tensor &idx, double scale, int64_t code, const Walk *walk) {
        const Tensor w = logits.detach(), probs = at::empty_like(w);
        Tensor y = forward_into(x, a, b, w, probs, (int) code, *walk);
        ctx->save_for_backward({x, a, b, probs, start, idx});
        ctx->saved_data["scale"] = scale;
        ctx->saved_data["code"] = code;
        if (!walk->tables.empty()) {
            ctx->saved_data["tables"] = walk->tables;
            ctx->saved_data["sizes"] = std::vector<int64_t>{walk->steps, walk->n_fix, walk->rows, walk->here, walk->weights};
        }
        return y;
    }

    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const variable_list saved = ctx->get_saved_variables();
        const int code = (int) ctx->saved_data["code"].toInt();
        check_saved(saved, [&](size_t) { return code; });
        const Tensor &x = saved[0], &a = saved[1], &b = saved[2], &probs = saved[3], &start = saved[4], &idx = saved[5];
        const double scale = ctx->saved_data["scale"].toDouble();
        Walk walk;
        const auto tables = ctx->saved_data.find("tables");
        if (tables != ctx->saved_data.end()) {
            walk.tables = tables->second.toTensorVector();
            const std::vector<int64_t> sizes = ctx->saved_data["sizes"].toIntVector();
            walk.steps = sizes[0], walk.n_fix = sizes[1], walk.rows = sizes[2], walk.here = sizes[3] != 0, walk.weights = sizes[4] != 0;
        }
        const c10::DeviceGuard guard(x.device());
        const Tensor gy = grads[0].contiguous();
        TORCH_CHECK(gy.scalar_type() == x.scalar_type() && gy.dim() == 2 && gy.size(0) == probs.size(0) && gy.size(1) == x.size(1)
                        && gy.device() == x.device(),
                    "expected grad_y [out,B] of x's dtype and device");
        const bool want_x = ctx->needs_input_grad(0), want_w = ctx->needs_input_grad(1);
        const int64_t in_dim = x.size(0), out_dim = probs.size(0), batch = x.size(1);
        const int64_t *ap = a.const_data_ptr<int64_t>(), *bp = b.const_data_ptr<int64_t>();
        // Along a schedule the one pass forms both gradients faster than the other kernels form grad_x alone (a task that asks for
        // x only, both wanting gradients: 128000 -> 128000 at batch 1024 349 / 470 us, 64000 at 512 94 / 104).
        const bool one_pass = want_x && !walk.tables.empty(), both = want_x && want_w;
        Tensor gx = want_x ? at::empty_like(x) : Tensor(), gw = want_w || one_pass ? at::empty_like(probs) : Tensor();
        int st = DL_ERR_TOO_LARGE;
        if (one_pass) {
            const int64_t bytes = dl_logic_backward_chained_workspace_bytes(walk.rows, out_dim, batch, code | DL_ROWS_ANY);
            check(bytes < 0 ? (int) -bytes : DL_OK, "logic_layer_cuda_backward_chained");
            const Tensor ws = bytes ? at::empty({bytes}, x.options().dtype(at::kByte)) : Tensor();
            st = dl_logic_backward_chained(x.const_data_ptr(), walk.i32(0), walk.i32(1), walk.flip(), walk.i32(3), walk.steps,
                                           probs.const_data_ptr(), gy.const_data_ptr(), 1,
                                           walk.n_fix ? walk.i32(4) : nullptr, walk.n_fix ? walk.i32(5) : nullptr, walk.n_fix,
                                           walk.rows, gw.mutable_data_ptr(), gx.mutable_data_ptr(),
                                           bytes ? ws.mutable_data_ptr() : nullptr, in_dim, out_dim, batch, scale,
                                           code | DL_ROWS_ANY | (walk.here ? DL_FIX_POSITIONS : 0), stream_of(x));
            if (st != DL_ERR_TOO_LARGE) check(st, "logic_layer_cuda_backward_chained");
        }
        if (st == DL_OK) {                                   // formed above
        } else if (both) {
            backward_both_into(x, a, b, probs, gy, start, idx, gw, gx, 0, scale, true, code);
        } else if (want_x) {
            check(dl_logic_backward_x(x.const_data_ptr(), ap, bp, probs.const_data_ptr(), gy.const_data_ptr(),
                                      start.const_data_ptr<int64_t>(), idx.const_data_ptr<int64_t>(), gx.mutable_data_ptr(),
                                      in_dim, out_dim, batch, scale, code, stream_of(x)),
                  "logic_layer_cuda_backward_x");
        } else if (want_w) {
            if (!walk.tables.empty() && walk.weights)
                st = dl_logic_backward_w_chained(x.const_data_ptr(), walk.i32(0), walk.i32(1), walk.flip(), walk.steps,
                                                 gy.const_data_ptr(), probs.const_data_ptr(), gw.mutable_data_ptr(), in_dim,
                                                 out_dim, batch, code | DL_ROWS_ANY, stream_of(x));
            if (st == DL_ERR_TOO_LARGE)
                st = dl_logic_backward_logits(x.const_data_ptr(), ap, bp, gy.const_data_ptr(), probs.const_data_ptr(),
                                              gw.mutable_data_ptr(), in_dim, out_dim, batch, code, stream_of(x));
            check(st, "logic_layer_cuda_backward_w");
        }
        return {gx, want_w ? gw : Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
    }
};

// Feature-major x and the layer's tensors as the kernels take them; the dtype code, or -1.
int layer_args(const Tensor &x, const Tensor &w, const Tensor &a, const Tensor &b) {
    if (!x.is_cuda() || x.dim() != 2 || w.dim() != 2 || w.size(1) != 16 || x.numel() == 0 || w.size(0) == 0) return -1;
    const c10::DeviceIndex device = x.get_device();
    if (!plain(w, device) || !index_of(a, device, w.size(0)) || !index_of(b, device, w.size(0))) return -1;
    return layer_code(x.scalar_type(), w.scalar_type());
}

bool reverse_args(const Tensor &start, const Tensor &idx, c10::DeviceIndex device, int64_t in_dim, int64_t out_dim) {
    return index_of(start, device, in_dim + 1) && index_of(idx, device, 2 * out_dim);
}

// A training layer on x [B, in] as LogicLayer.forward_cuda runs it: y [B, out], a view of [out, B].
c10::optional<Tensor> train_layer(const Tensor &x, const Tensor &weights, const Tensor &a, const Tensor &b, const Tensor &start,
                                  const Tensor &idx, double scale, std::vector<Tensor> tables, int64_t steps, int64_t n_fix,
                                  int64_t rows, bool here, bool walk_forward, bool walk_weights) {
    const int code = layer_args(x, weights, a, b);
    const Walk walk{std::move(tables), steps, n_fix, rows, here, walk_forward, walk_weights};
    if (code < 0 || !reverse_args(start, idx, x.get_device(), x.size(1), weights.size(0)) || !fits(walk, x.get_device()))
        return c10::nullopt;
    const c10::DeviceGuard guard(x.device());
    return LayerFunction::apply(x.transpose(0, 1).contiguous(), weights, a, b, start, idx, scale, (int64_t) code, &walk)
        .transpose(0, 1);
}

// A layer in eval mode on float x [B, in] (LogicLayer.forward_cuda): all of each neuron's argmax gate, no gradients.
// `tables`: verts, neuron and flip of the schedule that the kernel walks, or none.
c10::optional<Tensor> eval_layer(const Tensor &x, const Tensor &weights, const Tensor &a, const Tensor &b,
                                 const std::vector<Tensor> &tables, int64_t steps, int64_t in_dim) {
    const int code = layer_args(x, weights, a, b);
    if (code < 0 || x.size(1) != in_dim || (!tables.empty() && tables.size() != 3)) return c10::nullopt;
    for (size_t i = 0; i < tables.size(); ++i)
        if (tables[i].scalar_type() != (i == 2 ? at::kByte : at::kInt) || tables[i].numel() != steps + (i == 0)
            || !plain(tables[i], x.get_device()))
            return c10::nullopt;
    const at::NoGradGuard no_grad;
    const c10::DeviceGuard guard(x.device());
    const Tensor xt = x.transpose(0, 1).contiguous();
    const int64_t out_dim = weights.size(0), batch = xt.size(1);
    Tensor y = at::empty({out_dim, batch}, xt.options());
    int st = DL_ERR_TOO_LARGE;
    if (!tables.empty())
        st = dl_logic_forward_chained(xt.const_data_ptr(), tables[0].const_data_ptr<int32_t>(), tables[1].const_data_ptr<int32_t>(),
                                      tables[2].const_data_ptr<uint8_t>(), steps, weights.const_data_ptr(), y.mutable_data_ptr(),
                                      nullptr, in_dim, out_dim, batch, code | DL_GATES_OF_ARGMAX | DL_ROWS_ANY, stream_of(xt));
    if (st == DL_ERR_TOO_LARGE)
        st = dl_logic_forward(xt.const_data_ptr(), a.const_data_ptr<int64_t>(), b.const_data_ptr<int64_t>(), weights.const_data_ptr(),
                              y.mutable_data_ptr(), in_dim, out_dim, batch, code | DL_GATES_OF_ARGMAX, stream_of(xt));
    check(st, "logic_layer_cuda_forward");
    return y.transpose(0, 1);
}

// difflogic_cuda.forward_logits without a schedule.
c10::optional<std::tuple<Tensor, Tensor>> forward_logits(const Tensor &x, const Tensor &a, const Tensor &b, const Tensor &logits) {
    const int code = layer_args(x, logits, a, b);
    if (code < 0 || !x.is_contiguous()) return c10::nullopt;
    const c10::DeviceGuard guard(x.device());
    Tensor probs = at::empty_like(logits);
    Tensor y = forward_into(x, a, b, logits, probs, code, Walk());
    return std::make_tuple(y, probs);
}

// difflogic_cuda.backward_both; classes > 0: gy is the [classes, B] gradient of a GroupSum behind the layer.
c10::optional<std::tuple<Tensor, Tensor>> backward_both(const Tensor &x, const Tensor &a, const Tensor &b, const Tensor &w,
                                                        const Tensor &gy, const Tensor &start, const Tensor &idx, double scale,
                                                        bool softmax, int64_t classes) {
    const int code = layer_args(x, w, a, b);
    if (code < 0 || !x.is_contiguous() || !reverse_args(start, idx, x.get_device(), x.size(0), w.size(0))
        || !plain(gy, x.get_device()) || gy.dim() != 2 || gy.scalar_type() != x.scalar_type() || gy.size(1) != x.size(1)
        || gy.size(0) != (classes ? classes : w.size(0)) || classes < 0
        || (classes && (w.size(0) % classes || !softmax || w.scalar_type() != x.scalar_type())))
        return c10::nullopt;
    const c10::DeviceGuard guard(x.device());
    Tensor gw = at::empty_like(w), gx = at::empty_like(x);
    backward_both_into(x, a, b, w, gy, start, idx, gw, gx, classes, scale, softmax, code);
    return std::make_tuple(gw, gx);
}

// difflogic_cuda.backward_logits without a schedule.
c10::optional<Tensor> backward_logits(const Tensor &x, const Tensor &a, const Tensor &b, const Tensor &gy, const Tensor &probs) {
    const int code = layer_args(x, probs, a, b);
    if (code < 0 || !x.is_contiguous() || !plain(gy, x.get_device()) || gy.dim() != 2 || gy.scalar_type() != x.scalar_type()
        || gy.size(0) != probs.size(0) || gy.size(1) != x.size(1))
        return c10::nullopt;
    const c10::DeviceGuard guard(x.device());
    Tensor gw = at::empty_like(probs);
    check(dl_logic_backward_logits(x.const_data_ptr(), a.const_data_ptr<int64_t>(), b.const_data_ptr<int64_t>(),
                                   gy.const_data_ptr(), probs.const_data_ptr(), gw.mutable_data_ptr(), x.size(0), probs.size(0),
                                   x.size(1), code, stream_of(x)),
          "logic_layer_cuda_backward_logits");
    return gw;
}

// difflogic_cuda.forward_group_sum: (scores [B, k], probs).
c10::optional<std::tuple<Tensor, Tensor>> forward_group_sum(const Tensor &x, const Tensor &a, const Tensor &b, const Tensor &logits,
                                                            int64_t k, double tau) {
    const int code = layer_args(x, logits, a, b);
    if (code < 0 || x.scalar_type() != logits.scalar_type() || !x.is_contiguous() || k <= 0 || logits.size(0) % k)
        return c10::nullopt;
    const c10::DeviceGuard guard(x.device());
    Tensor y = at::empty({x.size(1), k}, x.options()), probs = at::empty_like(logits);
    const int64_t bytes = dl_group_sum_workspace_bytes(logits.size(0), x.size(1), k, code);
    const Tensor ws = at::empty({std::max<int64_t>(1, bytes)}, x.options().dtype(at::kByte));
    check(dl_logic_forward_group_sum(x.const_data_ptr(), a.const_data_ptr<int64_t>(), b.const_data_ptr<int64_t>(),
                                     logits.const_data_ptr(), probs.mutable_data_ptr(), y.mutable_data_ptr(),
                                     ws.mutable_data_ptr(), x.size(0), logits.size(0), x.size(1), k, tau, code, stream_of(x)),
          "logic_layer_cuda_forward_group_sum");
    return std::make_tuple(y, probs);
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

// LogicNetFunction's work for layers without schedules: all of a net's layers and its GroupSum, each way.  fused: the last layer and
// the GroupSum in one kernel each way (LogicLayerGroupSumFunction).
struct Net {
    std::vector<Tensor> a, b, start, idx;
    std::vector<double> scale;
    std::vector<int64_t> code;
    int64_t k = 0;
    double tau = 1.0;
    bool fused = false;
};

// Forward: (scores [B, k], what the backward pass needs: six tensors a layer).
std::tuple<Tensor, variable_list> net_forward_of(const Tensor &x, const variable_list &weights, const Net *net) {
    const size_t layers = net->a.size();
    variable_list saved;
    saved.reserve(6 * layers);
    Tensor cur = x;
    for (size_t l = 0; l < layers; ++l) {
        const Tensor w = weights[l].detach(), probs = at::empty_like(w);
        saved.insert(saved.end(), {cur, net->a[l], net->b[l], probs, net->start[l], net->idx[l]});
        if (l + 1 < layers || !net->fused) {
            cur = forward_into(cur, net->a[l], net->b[l], w, probs, (int) net->code[l], Walk());
            continue;
        }
        const int code = (int) net->code[l];
        const int64_t out_dim = w.size(0), batch = cur.size(1);
        Tensor y = at::empty({batch, net->k}, cur.options());
        const int64_t bytes = dl_group_sum_workspace_bytes(out_dim, batch, net->k, code);
        const Tensor ws = at::empty({std::max<int64_t>(1, bytes)}, cur.options().dtype(at::kByte));
        check(dl_logic_forward_group_sum(cur.const_data_ptr(), net->a[l].const_data_ptr<int64_t>(),
                                         net->b[l].const_data_ptr<int64_t>(), w.const_data_ptr(), probs.mutable_data_ptr(),
                                         y.mutable_data_ptr(), ws.mutable_data_ptr(), cur.size(0), out_dim, batch, net->k,
                                         net->tau, code, stream_of(cur)),
              "logic_layer_cuda_forward_group_sum");
        cur = y;
    }
    if (!net->fused) {
        const int code = layer_code(cur.scalar_type(), cur.scalar_type());
        const int64_t out_dim = cur.size(0), batch = cur.size(1);
        Tensor y = at::empty({batch, net->k}, cur.options());
        const int64_t bytes = dl_group_sum_workspace_bytes(out_dim, batch, net->k, code);
        const Tensor ws = at::empty({std::max<int64_t>(1, bytes)}, cur.options().dtype(at::kByte));
        check(dl_group_sum_forward(cur.const_data_ptr(), y.mutable_data_ptr(), ws.mutable_data_ptr(), out_dim, batch, net->k,
                                   net->tau, code, stream_of(cur)),
              "group_sum_forward");
        cur = y;
    }
    return {cur, saved};
}

// Backward, from the gradient of the scores: the gradients of x and the weights as `wanted`.  (A node's own checks have been
// made: saved is what net_forward returned.)
std::vector<c10::optional<Tensor>> net_backward(const variable_list &saved, Tensor g, const std::vector<bool> &wanted,
                                                const std::vector<double> &scale, const std::vector<int64_t> &codes, int64_t k,
                                                double tau, bool fused) {
    const int64_t layers = (int64_t) saved.size() / 6;
    TORCH_CHECK(layers > 0 && (int64_t) wanted.size() == layers + 1 && (int64_t) scale.size() == layers && (int64_t) codes.size() == layers,
                "net_backward: lists of one length expected");
    check_saved(saved, [&](size_t layer) { return codes[layer]; });
    const c10::DeviceGuard guard(saved[0].device());
    const Tensor &top = saved[6 * (layers - 1)];             // the last layer's input
    TORCH_CHECK(g.dim() == 2 && g.size(0) == top.size(1) && g.size(1) == k && g.scalar_type() == top.scalar_type()
                    && g.device() == top.device(),
                "expected the gradient of the scores [B,k] in their dtype and on their device");
    if (fused) {
        g = (g / tau).t().contiguous();                      // [k, B]: a few KB
    } else {
        g = g.contiguous();
        const int64_t out_dim = saved[6 * (layers - 1) + 3].size(0);
        Tensor gx = at::empty({out_dim, g.size(0)}, g.options());
        check(dl_group_sum_backward(g.const_data_ptr(), gx.mutable_data_ptr(), out_dim, g.size(0), k, tau,
                                    layer_code(g.scalar_type(), g.scalar_type()), stream_of(g)),
              "group_sum_backward");
        g = gx;
    }
    std::vector<c10::optional<Tensor>> out((size_t) layers + 1);       // of x, of the weights
    for (int64_t l = layers - 1; l >= 0; --l) {
        const Tensor *s = &saved[(size_t) (6 * l)];
        const Tensor &x = s[0], &a = s[1], &b = s[2], &probs = s[3], &start = s[4], &idx = s[5];
        bool want_x = wanted[0];
        for (int64_t below = 0; below < l; ++below) want_x = want_x || wanted[(size_t) (1 + below)];
        const bool want_w = wanted[(size_t) (1 + l)];
        const int64_t in_dim = x.size(0), out_dim = probs.size(0), batch = x.size(1);
        const int code = (int) codes[(size_t) l];
        const int64_t classes = fused && l == layers - 1 ? k : 0;
        const int64_t *ap = a.const_data_ptr<int64_t>(), *bp = b.const_data_ptr<int64_t>();
        const int64_t *sp = start.const_data_ptr<int64_t>(), *ip = idx.const_data_ptr<int64_t>();
        Tensor gx = want_x ? at::empty_like(x) : Tensor(), gw = want_w ? at::empty_like(probs) : Tensor();
        if (want_x && want_w)
            backward_both_into(x, a, b, probs, g, start, idx, gw, gx, classes, scale[(size_t) l], true, code);
        else if (want_x)
            check(classes ? dl_logic_backward_x_grouped(x.const_data_ptr(), ap, bp, probs.const_data_ptr(), g.const_data_ptr(), sp,
                                                        ip, gx.mutable_data_ptr(), in_dim, out_dim, batch, classes,
                                                        scale[(size_t) l], code, stream_of(x))
                          : dl_logic_backward_x(x.const_data_ptr(), ap, bp, probs.const_data_ptr(), g.const_data_ptr(), sp, ip,
                                                gx.mutable_data_ptr(), in_dim, out_dim, batch, scale[(size_t) l], code,
                                                stream_of(x)),
                  "logic_layer_cuda_backward_x");
        else if (want_w)
            check(classes ? dl_logic_backward_logits_grouped(x.const_data_ptr(), ap, bp, g.const_data_ptr(),
                                                             probs.const_data_ptr(), gw.mutable_data_ptr(), in_dim, out_dim,
                                                             batch, classes, code, stream_of(x))
                          : dl_logic_backward_logits(x.const_data_ptr(), ap, bp, g.const_data_ptr(), probs.const_data_ptr(),
                                                     gw.mutable_data_ptr(), in_dim, out_dim, batch, code, stream_of(x)),
                  "logic_layer_cuda_backward_w");
        if (want_w) out[(size_t) (1 + l)] = gw;
        if (!want_x) break;                                  // nothing below wants a gradient
        g = gx;
        if (l == 0 && wanted[0]) out[0] = gx;
    }
    return out;
}

// A net on feature-major x [in, B] (LogicNetFunction): scores, saved tensors and the layers' dtype codes.
c10::optional<std::tuple<Tensor, variable_list, std::vector<int64_t>>> net_forward(const Tensor &x, const variable_list &weights, std::vector<Tensor> a, std::vector<Tensor> b,
                                std::vector<Tensor> start, std::vector<Tensor> idx, std::vector<double> scale, int64_t k, double tau,
                                bool fused) {
    const size_t layers = weights.size();
    if (layers == 0 || a.size() != layers || b.size() != layers || start.size() != layers || idx.size() != layers
        || scale.size() != layers || k <= 0 || !x.is_contiguous())
        return c10::nullopt;
    Net net{std::move(a), std::move(b), std::move(start), std::move(idx), std::move(scale), {}, k, tau, fused};
    int64_t in_dim = x.dim() == 2 ? x.size(0) : 0;
    for (size_t l = 0; l < layers; ++l) {
        const int code = layer_args(x, weights[l], net.a[l], net.b[l]);
        if (code < 0 || !reverse_args(net.start[l], net.idx[l], x.get_device(), in_dim, weights[l].size(0))) return c10::nullopt;
        net.code.push_back(code);
        in_dim = weights[l].size(0);
    }
    if (in_dim % k || (fused && weights.back().scalar_type() != x.scalar_type())) return c10::nullopt;
    const c10::DeviceGuard guard(x.device());
    const at::NoGradGuard no_grad;
    auto [y, saved] = net_forward_of(x, weights, &net);
    return std::make_tuple(y, saved, net.code);
}

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
    check(dl_groupbitsum(b.const_data_ptr(), out.mutable_data_ptr<int32_t>(), b.size(0), b.size(1), 64, pad, k,
                         stream_of(b)),
          "groupbitsum");
    return out;
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    typedef py::call_guard<py::gil_scoped_release> unlocked;
    m.def("train_layer", &train_layer, unlocked());
    m.def("net_forward", &net_forward, unlocked());
    m.def("net_backward", &net_backward, unlocked());
    m.def("eval_layer", &eval_layer, unlocked());
    m.def("forward_logits", &forward_logits, unlocked());
    m.def("backward_both", &backward_both, unlocked());
    m.def("backward_logits", &backward_logits, unlocked());
    m.def("forward_group_sum", &forward_group_sum, unlocked());
    m.def("group_sum", &group_sum, unlocked());
    m.def("eval_weights", &eval_weights, unlocked());
    m.def("gate_ids_folded", &gate_ids_folded, unlocked());
    m.def("pack_rows", &pack_rows, unlocked());
    m.def("count_rows", &count_rows, unlocked());
}
