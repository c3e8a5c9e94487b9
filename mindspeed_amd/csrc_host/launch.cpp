// The kernel calls of ops/_kernels.py on plain device tensors in native code: outputs and workspaces from torch's
// allocator, the device made current, one call of the C ABI on the current stream.  The Python functions of the same names
// do the same through ctypes (and bracket the call for a Recorder); a function here returns None for what it does not
// take (a dtype the kernels do not know), which the caller then hands to the Python function for its error message.
//
// Why: small and routing-only layer steps are bound by the host, and of the 8 to 16 us of such a call less than 4 are the
// launch.  Host time per call, Python and here, us: grouped matmul 13.1 and 4.7, permute 15.5 and 6.3, unpermute 9.1 and 4.0,
// its gradient 11.0 and 4.9, SwiGLU 8.1 and 3.8; a small fp32 layer's training step 404 -> 271, routing layers of 4096 x 4096
// and 2731 x 2048 tokens, forward and backward, 178 -> 114 and 184 -> 120.
//
// Which ops: those that the steps of the index-form, routing-map and expert-module layers consist of.  The chunk sort (two
// calls of 82 and 88 us on the device at the size it is measured at, 16384 x 7168), one weight matrix per expert, the maps
// without rows and the SwiGLU backward in a matmul's epilogue stay with the Python functions alone.
//
// Below the calls: their autograd nodes, and the index-form layer and the routing-map permute and unpermute as chains of them.
// A Python node costs 5 to 15 us in each direction, and more where the scheduler puts the autograd thread on a core whose caches
// hold nothing of the interpreter: the figures in front of run_layer.
#include <dlfcn.h>
#include <torch/extension.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/TensorSubclassLikeUtils.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <atomic>
#include <optional>
#include <stdexcept>
#include <string>
#include <tuple>

#include "../../include/mindspeed_amd.h"
#include "../csrc/internal.h"

namespace {

namespace py = pybind11;
using at::Tensor;
using OptTensor = std::optional<Tensor>;

struct Api {
#define MS_API(name) decltype(&::name) name = nullptr;
    MS_API(ms_last_error)
    MS_API(ms_gmm_workspace_size)
    MS_API(ms_gmm_workspace_size_split)
    MS_API(ms_gmm)
    MS_API(ms_gmm_swiglu)
    MS_API(ms_moe_token_permute_workspace_size)
    MS_API(ms_moe_token_permute)
    MS_API(ms_moe_token_permute_grad)
    MS_API(ms_moe_token_unpermute)
    MS_API(ms_moe_routing_map_workspace_size)
    MS_API(ms_moe_routing_map_probs_grad)
    MS_API(ms_swiglu)
    MS_API(ms_swiglu_grad)
    MS_API(msi_routing_map_permute)
    MS_API(msi_unpermute_grad)
    MS_API(msi_gmm_backward_workspace_size)
    MS_API(msi_gmm_backward)
#undef MS_API
} api;

// What a failed call of the library becomes in Python (mindspeed_amd._lib.MindSpeedAmdError).
struct CallError : std::runtime_error {
    using std::runtime_error::runtime_error;
};
PyObject *error_class = nullptr;

// While a Recorder takes note of every op (flop_counter.record) the nodes' backward passes call the Python functions too.
std::atomic<bool> recording{false};
PyObject *device_fns = nullptr;                // op name -> Python function (ops/_kernels.py)
void record_through(py::dict fns) { device_fns = fns.release().ptr(); }
void set_recording(bool on) { recording = on; }

void bind(const std::string &path, py::object error) {
    void *lib = dlopen(path.c_str(), RTLD_NOW | RTLD_LOCAL);
    if (lib == nullptr) throw std::runtime_error(dlerror());
    auto find = [&](const char *name) {
        void *fn = dlsym(lib, name);
        if (fn == nullptr) throw std::runtime_error(path + " lacks " + name + ": rebuild it with `python -m mindspeed_amd.build`");
        return fn;
    };
    const std::string theirs = reinterpret_cast<decltype(&msi_interface)>(find("msi_interface"))();
    if (theirs != MS_INTERFACE)
        throw std::runtime_error("_host.so was built for entry points " MS_INTERFACE ", " + path + " has " + theirs +
                                 ": rebuild both with `python -m mindspeed_amd.build`");
#define MS_FIND(name) api.name = reinterpret_cast<decltype(&::name)>(find(#name));
    MS_FIND(ms_last_error)
    MS_FIND(ms_gmm_workspace_size)
    MS_FIND(ms_gmm_workspace_size_split)
    MS_FIND(ms_gmm)
    MS_FIND(ms_gmm_swiglu)
    MS_FIND(ms_moe_token_permute_workspace_size)
    MS_FIND(ms_moe_token_permute)
    MS_FIND(ms_moe_token_permute_grad)
    MS_FIND(ms_moe_token_unpermute)
    MS_FIND(ms_moe_routing_map_workspace_size)
    MS_FIND(ms_moe_routing_map_probs_grad)
    MS_FIND(ms_swiglu)
    MS_FIND(ms_swiglu_grad)
    MS_FIND(msi_routing_map_permute)
    MS_FIND(msi_unpermute_grad)
    MS_FIND(msi_gmm_backward_workspace_size)
    MS_FIND(msi_gmm_backward)
#undef MS_FIND
    error_class = error.release().ptr();
}

void check(int rc, const char *what) {
    if (rc != 0) throw CallError(std::string(what) + " failed (status " + std::to_string(rc) + "): " + api.ms_last_error());
}

// MS_* code of a dtype the kernels take, -1 otherwise.
int code(const Tensor &t) {
    switch (t.scalar_type()) {
        case at::kBFloat16: return MS_BF16;
        case at::kHalf: return MS_FP16;
        case at::kFloat: return MS_FP32;
        default: return -1;
    }
}
int code_or_zero(const OptTensor &t) { return t.has_value() ? code(*t) : 0; }
void *ptr(const Tensor &t) { return t.data_ptr(); }
void *ptr(const OptTensor &t) { return t.has_value() ? t->data_ptr() : nullptr; }

ms_stream_t stream_of(const Tensor &t) {
    return c10::hip::getCurrentHIPStream(t.device().index()).stream();
}
Tensor workspace(size_t bytes, const Tensor &like) {
    return at::empty({static_cast<int64_t>(bytes < 256 ? 256 : bytes)}, like.options().dtype(at::kByte));
}
Tensor none_of(const Tensor &like, at::ScalarType dtype) { return at::empty({0}, like.options().dtype(dtype)); }

// The kernels take probabilities in the tokens' dtype or in fp32; any other pair is widened to fp32 first, which is exact.
OptTensor kernel_probs(const OptTensor &probs, const Tensor &tokens) {
    if (!probs.has_value() || probs->scalar_type() == tokens.scalar_type() || probs->scalar_type() == at::kFloat) return probs;
    return probs->to(at::kFloat);
}

bool gmm_launch(const Tensor &x, const Tensor &w, const Tensor &gl, int64_t group_type, int64_t list_type, const Tensor &out,
                bool accumulate) {
    const int dtype = code(x);
    const bool rows = group_type == 0;
    const int64_t groups = gl.numel(), m = x.size(rows ? 0 : 1), k = x.size(rows ? 1 : 0), n = w.size(rows ? 2 : 1);
    const int out_dtype = out.scalar_type() == at::kFloat ? MS_FP32 : dtype;
    size_t bytes = 0;
    check(api.ms_gmm_workspace_size_split(groups, m, k, n, static_cast<int>(group_type), dtype, out_dtype, accumulate, &bytes),
          "ms_gmm_workspace_size_split");
    const Tensor ws = workspace(bytes, x);
    check(api.ms_gmm(stream_of(x), ptr(x), x.stride(0), x.stride(1), ptr(w), rows ? w.stride(0) : 0, w.stride(rows ? 1 : 0),
                     w.stride(rows ? 2 : 1), ptr(out), n, gl.const_data_ptr<int64_t>(), static_cast<int>(list_type),
                     static_cast<int>(group_type), groups, m, k, n, dtype, out_dtype, accumulate, ptr(ws), ws.numel()),
          "ms_gmm");
    return true;
}

OptTensor gmm(const Tensor &x, const Tensor &w, const Tensor &gl, int64_t group_type, int64_t list_type) {
    if (code(x) < 0) return {};
    const c10::DeviceGuard guard(x.device());
    const Tensor out = group_type == 0 ? at::empty({x.size(0), w.size(2)}, x.options())
                                       : at::empty({gl.numel(), x.size(0), w.size(1)}, x.options());
    gmm_launch(x, w, gl, group_type, list_type, out, false);
    return out;
}

bool gmm_out(const Tensor &x, const Tensor &w, const Tensor &gl, int64_t group_type, int64_t list_type, const Tensor &out,
             bool accumulate) {
    if (code(x) < 0) return false;
    const c10::DeviceGuard guard(x.device());
    return gmm_launch(x, w, gl, group_type, list_type, out, accumulate);
}

OptTensor gmm_backward(const Tensor &grad, const Tensor &x, const Tensor &w, const Tensor &gl, int64_t list_type, const Tensor &dw,
                       bool accumulate) {
    if (code(x) < 0) return {};
    const c10::DeviceGuard guard(x.device());
    const int64_t m = x.size(0), k = x.size(1), n = w.size(2), groups = gl.numel();
    const int dw_dtype = dw.scalar_type() == at::kFloat ? MS_FP32 : code(x);
    const Tensor dx = at::empty({m, k}, x.options());
    size_t bytes = 0;
    check(api.msi_gmm_backward_workspace_size(groups, m, k, n, code(x), dw_dtype, accumulate, &bytes), "msi_gmm_backward_workspace_size");
    const Tensor ws = workspace(bytes, x);
    check(api.msi_gmm_backward(stream_of(x), ptr(grad), grad.stride(0), grad.stride(1), ptr(x), x.stride(0), x.stride(1), ptr(w),
                               w.stride(0), w.stride(1), w.stride(2), ptr(dx), ptr(dw), gl.const_data_ptr<int64_t>(),
                               static_cast<int>(list_type), groups, m, k, n, code(x), dw_dtype, accumulate, ptr(ws), ws.numel()),
          "ms_gmm");
    return dx;
}

std::optional<std::tuple<Tensor, Tensor>> gmm_swiglu(const Tensor &x, const Tensor &w, const Tensor &gl, int64_t list_type,
                                                     const OptTensor &probs, bool want_fc1) {
    if (code(x) < 0 || code_or_zero(probs) < 0) return {};
    const c10::DeviceGuard guard(x.device());
    const int64_t m = x.size(0), k = x.size(1), ffn = w.size(2) / 2;
    const Tensor fc1 = want_fc1 ? at::empty({m, 2 * ffn}, x.options()) : none_of(x, x.scalar_type());
    const Tensor act = at::empty({m, ffn}, x.options());
    size_t bytes = 0;
    check(api.ms_gmm_workspace_size(gl.numel(), m, 0, &bytes), "ms_gmm_workspace_size");
    const Tensor ws = workspace(bytes, x);
    check(api.ms_gmm_swiglu(stream_of(x), ptr(x), x.stride(0), x.stride(1), ptr(w), w.stride(0), w.stride(1), w.stride(2),
                            want_fc1 ? ptr(fc1) : nullptr, 2 * ffn, ptr(act), ffn, ptr(probs), code_or_zero(probs),
                            gl.const_data_ptr<int64_t>(), static_cast<int>(list_type), gl.numel(), m, k, ffn, code(x), ptr(ws),
                            ws.numel()),
          "ms_gmm_swiglu");
    return std::make_tuple(fc1, act);
}

std::optional<std::tuple<Tensor, Tensor, Tensor, Tensor>> token_permute(const Tensor &tokens, const Tensor &indices, int64_t num_out,
                                                                        int64_t num_experts, bool want_sorted, bool want_counts) {
    const at::ScalarType it = indices.scalar_type();
    if (code(tokens) < 0 || (it != at::kLong && it != at::kInt)) return {};
    const c10::DeviceGuard guard(tokens.device());
    const int64_t num_tokens = tokens.size(0), hidden = tokens.size(1), topk = indices.dim() == 1 ? 1 : indices.size(1);
    const int64_t num_counts = want_counts && num_experts > 0 ? num_experts : 0;
    const auto ints = tokens.options().dtype(at::kInt);
    const Tensor row_id_map = at::empty({num_tokens * topk}, ints);
    const Tensor permuted = at::empty({num_out, hidden}, tokens.options());
    const Tensor sorted = at::empty({want_sorted ? num_out : 0}, ints);
    const Tensor counts = at::empty({num_counts}, tokens.options().dtype(at::kLong));
    size_t bytes = 0;
    check(api.ms_moe_token_permute_workspace_size(num_tokens, topk, num_experts, &bytes), "ms_moe_token_permute_workspace_size");
    const Tensor ws = workspace(bytes, tokens);
    check(api.ms_moe_token_permute(stream_of(tokens), ptr(tokens), ptr(indices), it == at::kLong ? MS_INT64 : MS_INT32, num_tokens,
                                   topk, hidden, code(tokens), num_out, num_experts, ptr(permuted), row_id_map.data_ptr<int32_t>(),
                                   want_sorted ? sorted.data_ptr<int32_t>() : nullptr,
                                   num_counts > 0 ? counts.data_ptr<int64_t>() : nullptr, ptr(ws), ws.numel()),
          "ms_moe_token_permute");
    return std::make_tuple(permuted, row_id_map, sorted, counts);
}

OptTensor token_permute_grad(const Tensor &grad, const Tensor &row_id_map, int64_t num_tokens, int64_t topk) {
    if (code(grad) < 0) return {};
    const c10::DeviceGuard guard(grad.device());
    const Tensor out = at::empty({num_tokens, grad.size(1)}, grad.options());
    check(api.ms_moe_token_permute_grad(stream_of(grad), ptr(grad), row_id_map.const_data_ptr<int32_t>(), num_tokens, topk,
                                        grad.size(1), code(grad), grad.size(0), ptr(out)),
          "ms_moe_token_permute_grad");
    return out;
}

OptTensor token_unpermute(const Tensor &permuted, const Tensor &row_id_map, const OptTensor &given_probs, int64_t num_tokens,
                          int64_t topk) {
    if (code(permuted) < 0 || code_or_zero(given_probs) < 0) return {};
    const c10::DeviceGuard guard(permuted.device());
    const OptTensor probs = kernel_probs(given_probs, permuted);
    const Tensor out = at::empty({num_tokens, permuted.size(1)}, permuted.options());
    check(api.ms_moe_token_unpermute(stream_of(permuted), ptr(permuted), row_id_map.const_data_ptr<int32_t>(), ptr(probs),
                                     code_or_zero(probs), num_tokens, topk, permuted.size(1), code(permuted), permuted.size(0),
                                     ptr(out)),
          "ms_moe_token_unpermute");
    return out;
}

std::optional<std::tuple<Tensor, Tensor>> token_unpermute_grad(const Tensor &permuted, const Tensor &grad_out,
                                                               const Tensor &row_id_map, const OptTensor &given_probs,
                                                               int64_t num_tokens, int64_t topk, int64_t rows,
                                                               const OptTensor &sorted_flat) {
    if (code(grad_out) < 0 || code_or_zero(given_probs) < 0) return {};
    const c10::DeviceGuard guard(grad_out.device());
    const OptTensor probs = kernel_probs(given_probs, grad_out);
    const Tensor grad_permuted = at::empty({rows, grad_out.size(1)}, grad_out.options());
    Tensor grad_probs = probs.has_value() ? at::empty_like(*probs) : none_of(grad_out, grad_out.scalar_type());
    const int64_t mapped = rows < num_tokens * topk ? rows : num_tokens * topk;
    const bool all_zero_first = rows > mapped;
    if (all_zero_first) grad_permuted.zero_();
    check(api.msi_unpermute_grad(stream_of(grad_out), probs.has_value() ? ptr(permuted) : nullptr, ptr(grad_out),
                                 row_id_map.const_data_ptr<int32_t>(), ptr(probs), code_or_zero(probs), num_tokens, topk,
                                 grad_out.size(1), code(grad_out), mapped,
                                 sorted_flat.has_value() && !all_zero_first ? sorted_flat->const_data_ptr<int32_t>() : nullptr,
                                 ptr(grad_permuted), probs.has_value() ? ptr(grad_probs) : nullptr),
          "ms_moe_token_unpermute_grad");
    if (given_probs.has_value() && grad_probs.scalar_type() != given_probs->scalar_type())
        grad_probs = grad_probs.to(given_probs->scalar_type());
    return std::make_tuple(grad_permuted, grad_probs);
}

OptTensor swiglu(const Tensor &x, const OptTensor &probs) {
    if (code(x) < 0 || code_or_zero(probs) < 0) return {};
    const c10::DeviceGuard guard(x.device());
    const int64_t rows = x.size(0), ffn = x.size(1) / 2;
    const Tensor y = at::empty({rows, ffn}, x.options());
    check(api.ms_swiglu(stream_of(x), ptr(x), ptr(probs), code_or_zero(probs), rows, ffn, code(x), ptr(y)), "ms_swiglu");
    return y;
}

std::optional<std::tuple<Tensor, Tensor>> swiglu_grad(const Tensor &g, const Tensor &x, const OptTensor &probs) {
    if (code(x) < 0 || code_or_zero(probs) < 0) return {};
    const c10::DeviceGuard guard(x.device());
    const int64_t rows = x.size(0), ffn = x.size(1) / 2;
    const Tensor gx = at::empty_like(x);
    const Tensor gp = probs.has_value() ? at::empty_like(*probs) : none_of(x, x.scalar_type());
    check(api.ms_swiglu_grad(stream_of(x), ptr(g), ptr(x), ptr(probs), code_or_zero(probs), rows, ffn, code(x), ptr(gx),
                             probs.has_value() ? ptr(gp) : nullptr),
          "ms_swiglu_grad");
    return std::make_tuple(gx, gp);
}

std::optional<std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor>> routing_map_permute_probs(const Tensor &tokens, const Tensor &map,
                                                                                            const OptTensor &probs, int64_t rows,
                                                                                            bool drop_and_pad) {
    if (code(tokens) < 0 || code_or_zero(probs) < 0) return {};
    const c10::DeviceGuard guard(tokens.device());
    const int64_t num_tokens = map.size(0), num_experts = map.size(1), hidden = tokens.size(1);
    const auto ints = tokens.options().dtype(at::kInt);
    const Tensor row_id_map = at::empty({num_tokens * num_experts}, ints);
    const Tensor sorted_flat = at::empty({rows}, ints);
    const Tensor permuted = at::empty({rows, hidden}, tokens.options());
    const Tensor permuted_probs = probs.has_value() ? at::empty({rows}, probs->options()) : none_of(tokens, at::kFloat);
    const Tensor ids = at::empty({rows}, tokens.options().dtype(at::kLong));
    size_t bytes = 0;
    check(api.ms_moe_routing_map_workspace_size(num_tokens, num_experts, drop_and_pad, &bytes), "ms_moe_routing_map_workspace_size");
    const Tensor ws = workspace(bytes, tokens);
    check(api.msi_routing_map_permute(stream_of(tokens), ptr(tokens), ptr(map), num_tokens, num_experts, hidden, code(tokens), rows,
                                      drop_and_pad, ptr(permuted), row_id_map.data_ptr<int32_t>(), sorted_flat.data_ptr<int32_t>(),
                                      nullptr, ptr(probs), code_or_zero(probs), probs.has_value() ? ptr(permuted_probs) : nullptr,
                                      ids.data_ptr<int64_t>(), ptr(ws), ws.numel()),
          "msi_routing_map_permute");
    return std::make_tuple(permuted, row_id_map, sorted_flat, permuted_probs, ids);
}

OptTensor routing_map_probs_grad(const Tensor &row_id_map, const Tensor &grad, int64_t num_tokens, int64_t num_experts) {
    if (code(grad) < 0) return {};
    const c10::DeviceGuard guard(grad.device());
    const Tensor out = at::empty({num_tokens, num_experts}, grad.options());
    check(api.ms_moe_routing_map_probs_grad(stream_of(grad), row_id_map.const_data_ptr<int32_t>(), row_id_map.numel(), ptr(grad),
                                            code(grad), grad.numel(), ptr(out)),
          "ms_moe_routing_map_probs_grad");
    return out;
}

// Whether a call may go straight to the kernels (ops/_kernels.py: _plain): no dispatch or function mode is active, and every
// tensor among the arguments is a plain one (or a parameter) on a device.
bool plain_argument(PyObject *a) {
    if (a == Py_None) return true;
    if (THPVariable_CheckExact(a)) return THPVariable_Unpack(a).is_cuda();
    if (PyList_Check(a) || PyTuple_Check(a)) {
        PyObject *items = PySequence_Fast(a, "");
        if (items == nullptr) throw py::error_already_set();
        bool ok = true;
        for (Py_ssize_t i = 0; ok && i < PySequence_Fast_GET_SIZE(items); ++i) ok = plain_argument(PySequence_Fast_GET_ITEM(items, i));
        Py_DECREF(items);
        return ok;
    }
    return !THPVariable_Check(a);
}
bool plain(py::handle args) {
    if (c10::impl::TorchDispatchModeTLS::stack_len() != 0 || at::impl::PythonTorchFunctionTLS::stack_len() != 0) return false;
    return plain_argument(args.ptr());
}

// ---- autograd nodes -----------------------------------------------------------------------------------------------
// What the Python autograd functions of the same ops do (ops/gmm.py, swiglu.py, npu_moe_token_permute.py,
// npu_moe_token_unpermute.py, moe_permute_mask_map.py), with the same tensors saved.
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;
const Tensor kNone;

// The Python function of an op, for a Recorder.  No Python object leaves it (the caller does not hold the interpreter's lock).
template <typename Result, typename... Args>
Result recorded(const char *name, Args &&...args) {
    static_assert(!std::is_base_of_v<py::handle, Result>, "it would be given back without the interpreter's lock");
    const py::gil_scoped_acquire gil;
    try {
        const py::object out = py::handle(device_fns)[name](std::forward<Args>(args)...);
        if constexpr (!std::is_void_v<Result>) return py::cast<Result>(out);
    } catch (py::error_already_set &e) {
        e.restore();
        python_error err;
        err.persist();
        throw err;
    }
}
// A backward pass whose failed calls reach the caller as the error that the forward pass raises (the engine knows only its own).
template <typename Body>
variable_list backward_of(const Body &body) {
    try {
        return body();
    } catch (const CallError &e) {
        const py::gil_scoped_acquire gil;
        PyErr_SetString(error_class, e.what());
        python_error err;
        err.persist();
        throw err;
    }
}

bool unit_stride(const Tensor &t) { return t.stride(-1) == 1 || t.stride(-2) == 1 || t.size(-1) <= 1 || t.size(-2) <= 1; }

struct PermuteNode : torch::autograd::Function<PermuteNode> {       // permuted rows, row map, rows per expert
    static variable_list forward(AutogradContext *ctx, const Tensor &tokens, const Tensor &indices, int64_t num_experts) {
        auto [permuted, row_id_map, sorted, counts] =
            *token_permute(tokens.contiguous(), indices.contiguous(), indices.numel(), num_experts, false, true);
        ctx->save_for_backward({row_id_map});
        ctx->saved_data["tokens"] = tokens.size(0);
        ctx->set_materialize_grads(false);
        ctx->mark_non_differentiable({row_id_map, counts});
        return {permuted, row_id_map, counts};
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        return backward_of([&]() -> variable_list {
            if (!grads[0].defined()) return {kNone, kNone, kNone};
            const Tensor row_id_map = ctx->get_saved_variables()[0], grad = grads[0].contiguous();
            const int64_t tokens = ctx->saved_data["tokens"].toInt(), topk = row_id_map.numel() / tokens;
            if (recording) return {recorded<Tensor>("moe_token_permute_grad", grad, row_id_map, tokens, topk), kNone, kNone};
            return {*token_permute_grad(grad, row_id_map, tokens, topk), kNone, kNone};
        });
    }
};

struct GmmNode : torch::autograd::Function<GmmNode> {
    static Tensor forward(AutogradContext *ctx, const Tensor &x, const Tensor &w, const Tensor &counts) {
        ctx->save_for_backward({x, w, counts});
        return *gmm(x, w, counts, 0, 1);
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        return backward_of([&]() -> variable_list {
            const variable_list saved = ctx->get_saved_variables();
            const Tensor &x = saved[0], &w = saved[1], &counts = saved[2];
            const Tensor grad = unit_stride(grads[0]) ? grads[0] : grads[0].contiguous();
            const bool want_x = ctx->needs_input_grad(0), want_w = ctx->needs_input_grad(1);
            Tensor dx, dw;
            if (want_w) dw = at::empty(w.sizes(), x.options());
            if (want_x && want_w) {
                dx = recording ? recorded<Tensor>("gmm_backward", grad, x, w, counts, 1, dw, false) : *gmm_backward(grad, x, w, counts, 1, dw, false);
            } else if (want_w) {
                if (recording) recorded<void>("gmm_out", x.t(), grad, counts, 2, 1, dw, false);
                else gmm_out(x.t(), grad, counts, 2, 1, dw, false);
            } else if (want_x) {
                dx = recording ? recorded<Tensor>("gmm", grad, w.transpose(1, 2), counts, 0, 1) : *gmm(grad, w.transpose(1, 2), counts, 0, 1);
            }
            return {dx, dw, kNone};
        });
    }
};

struct SwigluNode : torch::autograd::Function<SwigluNode> {
    static Tensor forward(AutogradContext *ctx, const Tensor &x) {
        ctx->save_for_backward({x});
        return *swiglu(x, {});
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        return backward_of([&]() -> variable_list {
            const Tensor x = ctx->get_saved_variables()[0], grad = grads[0].contiguous();
            if (recording) return {std::get<0>(recorded<std::tuple<Tensor, Tensor>>("swiglu_grad", grad, x, OptTensor{}))};
            return {std::get<0>(*swiglu_grad(grad, x, {}))};
        });
    }
};

struct UnpermuteNode : torch::autograd::Function<UnpermuteNode> {
    static Tensor forward(AutogradContext *ctx, const Tensor &permuted, const Tensor &row_id_map, const Tensor &given_probs) {
        const Tensor probs = given_probs.contiguous();
        ctx->save_for_backward({permuted, row_id_map, probs});
        return *token_unpermute(permuted, row_id_map, probs, probs.size(0), probs.size(1));
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        return backward_of([&]() -> variable_list {
            const variable_list saved = ctx->get_saved_variables();
            const Tensor &permuted = saved[0], &row_id_map = saved[1], &probs = saved[2], grad = grads[0].contiguous();
            const int64_t tokens = probs.size(0), topk = probs.size(1), rows = permuted.size(0);
            const auto [d_permuted, d_probs] = recording
                ? recorded<std::tuple<Tensor, Tensor>>("moe_token_unpermute_grad", permuted, grad, row_id_map, probs, tokens, topk, rows)
                : *token_unpermute_grad(permuted, grad, row_id_map, probs, tokens, topk, rows, {});
            return {d_permuted, kNone, d_probs};
        });
    }
};

struct MapPermuteNode : torch::autograd::Function<MapPermuteNode> {  // what routing_map_permute_probs returns
    static variable_list forward(AutogradContext *ctx, const Tensor &tokens, const Tensor &map, const OptTensor &given_probs, int64_t rows,
                                 bool drop_and_pad) {
        const OptTensor probs = given_probs.has_value() ? OptTensor(given_probs->contiguous()) : given_probs;
        auto [permuted, row_id_map, sorted_flat, permuted_probs, ids] =
            *routing_map_permute_probs(tokens.contiguous(), map.contiguous(), probs, rows, drop_and_pad);
        ctx->save_for_backward({row_id_map});
        ctx->saved_data["tokens"] = map.size(0);
        ctx->set_materialize_grads(false);
        variable_list fixed{row_id_map, sorted_flat, ids};
        if (!probs.has_value()) fixed.push_back(permuted_probs);
        ctx->mark_non_differentiable(fixed);
        return {permuted, row_id_map, sorted_flat, permuted_probs, ids};
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        return backward_of([&]() -> variable_list {
            const Tensor row_id_map = ctx->get_saved_variables()[0];
            const int64_t tokens = ctx->saved_data["tokens"].toInt(), experts = row_id_map.numel() / tokens;
            Tensor d_tokens, d_probs;
            if (grads[0].defined() && ctx->needs_input_grad(0)) {
                const Tensor grad = grads[0].contiguous();
                d_tokens = recording ? recorded<Tensor>("moe_token_permute_grad", grad, row_id_map, tokens, experts)
                                     : *token_permute_grad(grad, row_id_map, tokens, experts);
            }
            if (grads[3].defined() && ctx->needs_input_grad(2)) {
                const Tensor grad = grads[3].contiguous();
                d_probs = recording ? recorded<Tensor>("routing_map_probs_grad", row_id_map, grad, tokens, experts)
                                    : *routing_map_probs_grad(row_id_map, grad, tokens, experts);
            }
            return {d_tokens, kNone, d_probs, kNone, kNone};
        });
    }
};

struct MapUnpermuteNode : torch::autograd::Function<MapUnpermuteNode> {
    static Tensor forward(AutogradContext *ctx, const Tensor &given, const Tensor &row_id_map, const Tensor &sorted_flat,
                          const OptTensor &given_probs, int64_t tokens, bool drop_and_pad) {
        const Tensor permuted = given.contiguous();
        const OptTensor probs = given_probs.has_value() ? OptTensor(given_probs->contiguous()) : given_probs;
        ctx->save_for_backward({probs.has_value() ? permuted : kNone, row_id_map, probs.has_value() ? *probs : kNone, sorted_flat});
        ctx->saved_data["tokens"] = tokens;
        ctx->saved_data["rows"] = permuted.size(0);
        ctx->saved_data["all_mapped"] = drop_and_pad;         // (every expert's capacity rows are filled)
        return *token_unpermute(permuted, row_id_map, probs, tokens, row_id_map.numel() / tokens);
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        return backward_of([&]() -> variable_list {
            const variable_list saved = ctx->get_saved_variables();
            const Tensor &row_id_map = saved[1], grad = grads[0].contiguous();
            const OptTensor probs = saved[2].defined() ? OptTensor(saved[2]) : OptTensor();
            const Tensor permuted = probs.has_value() ? saved[0] : at::empty({0}, grad.options());
            const OptTensor marked = ctx->saved_data["all_mapped"].toBool() ? OptTensor() : OptTensor(saved[3]);
            const int64_t tokens = ctx->saved_data["tokens"].toInt(), rows = ctx->saved_data["rows"].toInt();
            const int64_t experts = row_id_map.numel() / tokens;
            const auto [d_permuted, d_probs] = recording
                ? recorded<std::tuple<Tensor, Tensor>>("moe_token_unpermute_grad", permuted, grad, row_id_map, probs, tokens, experts, rows, marked)
                : *token_unpermute_grad(permuted, grad, row_id_map, probs, tokens, experts, rows, marked);
            return {d_permuted, kNone, kNone, probs.has_value() && ctx->needs_input_grad(3) ? d_probs : kNone, kNone, kNone};
        });
    }
};

// Whether nothing but autograd wants to see a call: no dispatch or function mode, no functorch transform, no tracer.
bool only_autograd() {
    const c10::DispatchKeySet keys = c10::impl::tls_local_dispatch_key_set().included_;
    return c10::impl::TorchDispatchModeTLS::stack_len() == 0 && at::impl::PythonTorchFunctionTLS::stack_len() == 0 &&
           !keys.has(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) && !keys.has(c10::DispatchKey::FuncTorchDynamicLayerBackMode) &&
           !torch::jit::tracer::isTracing();
}
// A plain tensor (or parameter) on a device, neither a dual number nor wrapped, with something in it; nullptr for anything else.
const Tensor *plain_tensor(py::handle h) {
    if (!THPVariable_CheckExact(h.ptr())) return nullptr;
    const Tensor &t = THPVariable_Unpack(h.ptr());
    if (!t.is_cuda() || t.layout() != at::kStrided || t.numel() == 0 || at::isTensorSubclassLike(t) || t._fw_grad(0).defined()) return nullptr;
    return &t;
}
bool takes(const Tensor &t) { return code(t) >= 0; }
bool fits16(const Tensor &t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }

// The functions below return None for a call that they do not take (a shape, type or layout that needs a look, a mistake, a
// transform): the Python functions then do, with their error messages.

// us per pass, forward and backward, with Python nodes and with these, where the scheduler puts the two threads well and where
// not (which lasts for a process): 512 tokens x 256 over 8 experts in fp32 149 and 275 -> 93 and 142; routing map of 4096 x 4096
// over 8 experts 84 and 115 -> 83 and 83 (84 on the device), 2731 x 2048 over 60 67 and 120 -> 64 and 87 (66 on the device).
// What is left beside the launches is the hand-over to the autograd thread and back.

// dispatcher.dispatch_mlp_combine without gradient fusion; fused: as inference runs it (activation in the first matmul's
// epilogue where the operands allow it, nothing kept).
Tensor run_layer(const Tensor &x, const Tensor &index, const Tensor &probs, const Tensor &w1, const Tensor &w2, int64_t experts,
                    bool fused) {
    if (!fused) {
        const variable_list permuted = PermuteNode::apply(x, index, experts);
        const Tensor act = SwigluNode::apply(GmmNode::apply(permuted[0], w1, permuted[2]));
        return UnpermuteNode::apply(GmmNode::apply(act, w2, permuted[2]), permuted[1], probs);
    }
    auto [permuted, row_id_map, sorted, counts] = *token_permute(x.contiguous(), index.contiguous(), index.numel(), experts, false, true);
    const int64_t hidden = x.size(1), ffn = w2.size(1);
    Tensor act;
    if (x.scalar_type() != at::kFloat && hidden % 8 == 0 && ffn % 8 == 0 && w2.size(2) % 8 == 0 && fits16(permuted) && fits16(w1) && fits16(w2))
        act = std::get<1>(*gmm_swiglu(permuted, w1, counts, 1, {}, false));
    else
        act = *swiglu(*gmm(permuted, w1, counts, 0, 1), {});
    const Tensor out = *gmm(act, w2, counts, 0, 1);
    return *token_unpermute(out, row_id_map, probs.contiguous(), probs.size(0), probs.size(1));
}
py::object layer(py::handle x_, py::handle index_, py::handle probs_, py::handle w1_, py::handle w2_, int64_t experts, bool fused) {
    if (!only_autograd()) return py::none();
    const Tensor *x = plain_tensor(x_), *index = plain_tensor(index_), *probs = plain_tensor(probs_), *w1 = plain_tensor(w1_),
                 *w2 = plain_tensor(w2_);
    if (x == nullptr || index == nullptr || probs == nullptr || w1 == nullptr || w2 == nullptr) return py::none();
    for (const Tensor *t : {index, probs, w1, w2})
        if (t->device() != x->device()) return py::none();
    const at::ScalarType it = index->scalar_type();
    if (!takes(*x) || !takes(*probs) || (it != at::kLong && it != at::kInt) || w1->scalar_type() != x->scalar_type() ||
        w2->scalar_type() != x->scalar_type() || x->dim() != 2 || (index->dim() != 1 && index->dim() != 2) || probs->dim() != 2 ||
        w1->dim() != 3 || w2->dim() != 3)
        return py::none();
    const int64_t topk = index->dim() == 1 ? 1 : index->size(1);
    if (index->size(0) != x->size(0) || probs->size(0) != x->size(0) || probs->size(1) != topk || experts < 1 || experts > 1024 ||
        w1->size(0) != experts || w1->size(1) != x->size(1) || w1->size(2) % 2 != 0 || w2->size(0) != experts ||
        w2->size(1) != w1->size(2) / 2 || !unit_stride(*w1) || !unit_stride(*w2) ||
        (fused && (at::GradMode::is_enabled() || !w1->is_contiguous())))
        return py::none();
    Tensor y;
    {
        const py::gil_scoped_release no_gil;
        y = run_layer(*x, *index, *probs, *w1, *w2, experts, fused);
    }
    return py::cast(y);
}

// (permuted rows, row map, flat positions, permuted probabilities or None, token numbers) of a routing map, and the rows asked for
py::object map_permute(py::handle tokens_, py::handle map_, py::handle probs_, py::handle rows_, bool drop_and_pad) {
    if (!only_autograd() || !PyLong_CheckExact(rows_.ptr())) return py::none();
    const Tensor *tokens = plain_tensor(tokens_), *map = plain_tensor(map_), *probs = probs_.is_none() ? nullptr : plain_tensor(probs_);
    if (tokens == nullptr || map == nullptr || (probs == nullptr && !probs_.is_none())) return py::none();
    if (!takes(*tokens) || tokens->dim() != 2 || map->dim() != 2 || map->scalar_type() != at::kBool || map->size(0) != tokens->size(0) ||
        map->device() != tokens->device() ||
        (probs != nullptr && (!takes(*probs) || probs->sizes() != map->sizes() || probs->device() != tokens->device())))
        return py::none();
    const int64_t experts = map->size(1);
    int64_t rows = PyLong_AsLongLong(rows_.ptr());
    if (rows == -1 && PyErr_Occurred() != nullptr) {
        PyErr_Clear();
        return py::none();
    }
    if (rows < 0 || rows > map->numel()) return py::none();
    if (drop_and_pad) rows = rows / experts * experts;
    variable_list out;
    {
        const py::gil_scoped_release no_gil;
        out = MapPermuteNode::apply(*tokens, *map, probs != nullptr ? OptTensor(*probs) : OptTensor(), rows, drop_and_pad);
    }
    return py::make_tuple(out[0], out[1], out[2], probs != nullptr ? py::cast(out[3]) : py::none(), out[4], rows);
}

// ... and back, by the row map and flat positions of that very map
py::object map_unpermute(py::handle permuted_, py::handle row_id_map_, py::handle sorted_flat_, py::handle probs_, py::handle map_,
                         int64_t tokens, bool drop_and_pad) {
    if (!only_autograd()) return py::none();
    const Tensor *permuted = plain_tensor(permuted_), *row_id_map = plain_tensor(row_id_map_), *sorted_flat = plain_tensor(sorted_flat_),
                 *map = plain_tensor(map_), *probs = probs_.is_none() ? nullptr : plain_tensor(probs_);
    if (permuted == nullptr || row_id_map == nullptr || sorted_flat == nullptr || map == nullptr || (probs == nullptr && !probs_.is_none()))
        return py::none();
    for (const Tensor *t : {row_id_map, sorted_flat, map})
        if (t->device() != permuted->device()) return py::none();
    if (!takes(*permuted) || permuted->dim() != 2 || map->dim() != 2 || map->scalar_type() != at::kBool || map->size(0) != tokens ||
        row_id_map->numel() != map->numel() || sorted_flat->numel() != permuted->size(0) ||
        (probs != nullptr && (!takes(*probs) || probs->sizes() != map->sizes() || probs->device() != permuted->device())))
        return py::none();
    Tensor y;
    {
        const py::gil_scoped_release no_gil;
        y = MapUnpermuteNode::apply(*permuted, *row_id_map, *sorted_flat, probs != nullptr ? OptTensor(*probs) : OptTensor(), tokens, drop_and_pad);
    }
    return py::cast(y);
}

}  // namespace

PYBIND11_MODULE(_host, mod) {
    py::register_exception_translator([](std::exception_ptr p) {
        try {
            if (p) std::rethrow_exception(p);
        } catch (const CallError &e) {
            PyErr_SetString(error_class != nullptr ? error_class : PyExc_RuntimeError, e.what());
        }
    });
    mod.def("bind", &bind);
    mod.def("plain", &plain);
    mod.def("record_through", &record_through);
    mod.def("set_recording", &set_recording);
    mod.def("layer", &layer);
    mod.def("map_permute", &map_permute);
    mod.def("map_unpermute", &map_unpermute);
    const py::call_guard<py::gil_scoped_release> no_gil;      // (a launch may wait for a full queue)
    mod.def("gmm", &gmm, no_gil);
    mod.def("gmm_out", &gmm_out, no_gil);
    mod.def("gmm_backward", &gmm_backward, no_gil);
    mod.def("gmm_swiglu", &gmm_swiglu, no_gil);
    mod.def("moe_token_permute", &token_permute, no_gil);
    mod.def("moe_token_permute_grad", &token_permute_grad, no_gil);
    mod.def("moe_token_unpermute", &token_unpermute, no_gil);
    mod.def("moe_token_unpermute_grad", &token_unpermute_grad, py::arg("permuted"), py::arg("grad_out"), py::arg("row_id_map"),
            py::arg("probs"), py::arg("num_tokens"), py::arg("topk"), py::arg("num_rows"), py::arg("sorted_flat") = py::none(), no_gil);
    mod.def("swiglu", &swiglu, no_gil);
    mod.def("swiglu_grad", &swiglu_grad, no_gil);
    mod.def("routing_map_permute_probs", &routing_map_permute_probs, no_gil);
    mod.def("routing_map_probs_grad", &routing_map_probs_grad, no_gil);
}
