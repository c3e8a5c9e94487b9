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
#include <dlfcn.h>
#include <torch/extension.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

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
