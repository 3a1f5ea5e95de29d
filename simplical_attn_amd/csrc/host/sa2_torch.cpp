// The operator's host path in native code: argument checks, output and workspace allocation, the calls of the C ABI
// (include/sa2.h) and the autograd formula, so that a call from Python costs one crossing into C++ each way and the
// backward runs in the autograd engine's thread without entering Python.
//
// What bounds a small call is this path.  Built in Python (checks, torch.empty, ctypes arrays, a Python autograd
// Function) B2 N256 H4 D64 w 32/32 took 217 us of host time for a forward and backward whose kernels take 106 us.
//
// The C ABI functions are handed over as addresses by bind(), so that the library is whichever one Python loaded.
// A call whose arguments this file does not accept goes to the Python checks, which raise the error that names them.
#include <ATen/TensorSubclassLikeUtils.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/extension.h>

#include <cmath>
#include <optional>

#include "sa2.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

decltype(&sa2_forward_ws) fwd_fn = nullptr;
decltype(&sa2_fwd_workspace_bytes) fwd_ws_fn = nullptr;
decltype(&sa2_backward) bwd_fn = nullptr;
decltype(&sa2_bwd_workspace_bytes) ws_fn = nullptr;
decltype(&sa2_strerror) err_fn = nullptr;

// A negative status of the C ABI; becomes simplical_attn_amd._lib.Sa2Error in Python
struct Status : std::runtime_error {
    int code;
    explicit Status(int c) : std::runtime_error("sa2 error " + std::to_string(c) + ": " + err_fn(c)), code(c) {}
};
void check(int rc) {
    if (rc != 0) throw Status(rc);
}

struct Args {
    int64_t w1, w2;
    double scale, k2_bias, v2_bias;
    bool inclusive;
    unsigned flags;
};

int dtype_code(const Tensor& t) {
    switch (t.scalar_type()) {
        case at::kFloat: return SA2_F32;
        case at::kBFloat16: return SA2_BF16;
        case at::kHalf: return SA2_F16;
        default: return -1;
    }
}
bool same(const Tensor& t, const Tensor& q) {
    return t.defined() && t.scalar_type() == q.scalar_type() && t.sizes() == q.sizes() && t.device() == q.device();
}
bool inputs_ok(const Tensor& q, const Tensor& k1, const Tensor& k2, const Tensor& v1, const Tensor& v2) {
    return q.dim() == 4 && dtype_code(q) >= 0 && q.is_cuda() && same(k1, q) && same(k2, q) && same(v1, q) && same(v2, q);
}
bool saved_ok(const Tensor& q, const Tensor& out, const Tensor& lse, const Tensor& dout) {
    return same(out, q) && same(dout, q) && lse.defined() && lse.scalar_type() == at::kFloat && lse.device() == q.device() && lse.dim() == 3 &&
           lse.size(0) == q.size(0) && lse.size(1) == q.size(2) && lse.size(2) == q.size(1) && lse.is_contiguous();
}

// Unit stride along head_dim and a positive stride on every axis longer than 1; anything else (broadcast views among
// it) is copied.
Tensor rows(const Tensor& t) {
    bool ok = t.stride(3) == 1;
    for (int a = 0; a < 3; ++a) ok = ok && (t.stride(a) > 0 || t.size(a) == 1);
    return ok ? t : t.contiguous();
}
void put_strides(int64_t* s, const Tensor& t) {
    s[0] = t.stride(0);
    s[1] = t.stride(1);
    s[2] = t.stride(2);
}

std::pair<Tensor, Tensor> run_forward(const Tensor& q_, const Tensor& k1_, const Tensor& k2_, const Tensor& v1_, const Tensor& v2_, const Args& a) {
    const Tensor q = rows(q_), k1 = rows(k1_), k2 = rows(k2_), v1 = rows(v1_), v2 = rows(v2_);
    const c10::DeviceGuard guard(q.device());
    const int64_t B = q.size(0), N = q.size(1), H = q.size(2), D = q.size(3);
    Tensor out = at::empty({B, N, H, D}, q.options().requires_grad(false));
    Tensor lse = at::empty({B, H, N}, q.options().dtype(at::kFloat).requires_grad(false));
    const size_t bytes = fwd_ws_fn((int)B, (int)N, (int)H, (int)D, (int)a.w1, (int)a.w2, dtype_code(q), a.inclusive ? 1 : 0, a.flags);
    const Tensor ws = bytes ? at::empty({(int64_t)bytes}, lse.options().dtype(at::kByte)) : Tensor();
    int64_t s[3 * SA2_FWD_TENSORS];
    const Tensor* const t[SA2_FWD_TENSORS] = {&q, &k1, &k2, &v1, &v2, &out};
    for (int i = 0; i < SA2_FWD_TENSORS; ++i) put_strides(s + 3 * i, *t[i]);
    check(fwd_fn(q.data_ptr(), k1.data_ptr(), k2.data_ptr(), v1.data_ptr(), v2.data_ptr(), out.data_ptr(), (float*)lse.data_ptr(),
                 bytes ? ws.data_ptr() : nullptr, bytes, (int)B, (int)N, (int)H, (int)D, s, (int)a.w1, (int)a.w2, (float)a.scale, (float)a.k2_bias, (float)a.v2_bias, dtype_code(q), a.inclusive ? 1 : 0,
                 a.flags, (void*)c10::hip::getCurrentHIPStream(q.device().index()).stream()));
    return {out, lse};
}

// `needs`: bit t set = gradient t of (q, k1, k2, v1, v2) is wanted; the others stay undefined
std::array<Tensor, 5> run_backward(const Tensor& q_, const Tensor& k1_, const Tensor& k2_, const Tensor& v1_, const Tensor& v2_, const Tensor& out_,
                                   const Tensor& lse, const Tensor& dout_, unsigned needs, const Args& a) {
    const Tensor q = rows(q_), k1 = rows(k1_), k2 = rows(k2_), v1 = rows(v1_), v2 = rows(v2_), out = rows(out_), dout = rows(dout_);
    const c10::DeviceGuard guard(q.device());
    const int64_t B = q.size(0), N = q.size(1), H = q.size(2), D = q.size(3);
    const int code = dtype_code(q), closed = a.inclusive ? 1 : 0;
    std::array<Tensor, 5> g;
    const auto like = q.options().requires_grad(false);
    for (int i = 0; i < 5; ++i)
        if (needs >> i & 1) g[i] = at::empty({B, N, H, D}, like);
    const size_t bytes = ws_fn((int)B, (int)N, (int)H, (int)D, (int)a.w1 - 1 + closed, (int)a.w2 - 1 + closed, code, a.flags);
    const Tensor ws = at::empty({(int64_t)std::max<size_t>(bytes, 256)}, like.dtype(at::kByte));
    int64_t s[3 * SA2_BWD_TENSORS];
    const Tensor* const t[7] = {&q, &k1, &k2, &v1, &v2, &out, &dout};
    for (int i = 0; i < 7; ++i) put_strides(s + 3 * i, *t[i]);
    for (int i = 0; i < 5; ++i) put_strides(s + 3 * (7 + i), g[i].defined() ? g[i] : q);
    auto ptr = [&](int i) { return g[i].defined() ? g[i].data_ptr() : nullptr; };
    check(bwd_fn(q.data_ptr(), k1.data_ptr(), k2.data_ptr(), v1.data_ptr(), v2.data_ptr(), out.data_ptr(), dout.data_ptr(),
                 (const float*)lse.data_ptr(), ptr(0), ptr(1), ptr(2), ptr(3), ptr(4), ws.data_ptr(), (size_t)ws.numel(), (int)B, (int)N, (int)H,
                 (int)D, s, (int)a.w1, (int)a.w2, (float)a.scale, (float)a.k2_bias, (float)a.v2_bias, code, closed, a.flags,
                 (void*)c10::hip::getCurrentHIPStream(q.device().index()).stream()));
    return g;
}

// Forward saves (q, k1, k2, v1, v2, out, LSE) and backward returns the five gradients (simplicial/triton_impl.py:54, 158).
struct Attention : torch::autograd::Function<Attention> {
    static Tensor forward(AutogradContext* ctx, const Tensor& q, const Tensor& k1, const Tensor& k2, const Tensor& v1, const Tensor& v2, Args a) {
        at::AutoDispatchBelowADInplaceOrView below;
        auto [out, lse] = run_forward(q, k1, k2, v1, v2, a);
        ctx->save_for_backward({q, k1, k2, v1, v2, out, lse});
        auto& d = ctx->saved_data;
        d["w1"] = a.w1;
        d["w2"] = a.w2;
        d["scale"] = a.scale;
        d["k2_bias"] = a.k2_bias;
        d["v2_bias"] = a.v2_bias;
        d["inclusive"] = a.inclusive;
        d["flags"] = (int64_t)a.flags;
        return out;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        at::AutoDispatchBelowADInplaceOrView below;
        const auto s = ctx->get_saved_variables();
        auto& d = ctx->saved_data;
        const Args a{d["w1"].toInt(),           d["w2"].toInt(),        d["scale"].toDouble(),          d["k2_bias"].toDouble(),
                     d["v2_bias"].toDouble(), d["inclusive"].toBool(), (unsigned)d["flags"].toInt()};
        unsigned needs = 0;
        for (int i = 0; i < 5; ++i) needs |= (ctx->needs_input_grad(i) ? 1u : 0u) << i;
        auto g = run_backward(s[0], s[1], s[2], s[3], s[4], s[5], s[6], grads[0], needs, a);
        return {g[0], g[1], g[2], g[3], g[4], Tensor()};
    }
};

double scale_of(const std::optional<double>& scale, const Tensor& q) { return scale ? *scale : 1.0 / std::sqrt((double)q.size(3)); }

// The Python checks (set by bind), which raise for arguments that inputs_ok / saved_ok refuse
PyObject *check_inputs_py = nullptr, *check_saved_py = nullptr;
void refuse_inputs(const Tensor& q, const Tensor& k1, const Tensor& k2, const Tensor& v1, const Tensor& v2) {
    py::handle checks{check_inputs_py};
    checks(q, k1, k2, v1, v2);
    throw std::invalid_argument("q, k1, k2, v1 and v2 must be GPU tensors of one shape [batch, seq_len, num_heads, head_dim], dtype and device");
}

// Calls that need more of autograd or of the dispatcher than the native formula gives go through the Python autograd
// function (set by bind):
//  - a tensor with a forward-mode tangent, for which the Python function raises (the native path below would drop the
//    tangent where no input requires grad, which reads as a zero derivative);
//  - a call under torch.jit.trace, which records the Python function as one operation (of the native path it would see
//    the allocation of the output only, and a replay would return uninitialised memory);
//  - tensors of torch.func transforms and other wrappers, and active dispatch modes.
PyObject* general_py = nullptr;
bool plain(const Tensor& t) { return !t._fw_grad(0).defined() && !at::isTensorSubclassLike(t); }

Tensor attention(const Tensor& q, const Tensor& k1, const Tensor& k2, const Tensor& v1, const Tensor& v2, int64_t w1, int64_t w2,
                 std::optional<double> scale, double k2_bias, double v2_bias, bool inclusive, unsigned flags) {
    if (!inputs_ok(q, k1, k2, v1, v2)) refuse_inputs(q, k1, k2, v1, v2);
    if (torch::jit::tracer::isTracing() || !(plain(q) && plain(k1) && plain(k2) && plain(v1) && plain(v2)))
        return py::handle{general_py}(q, k1, k2, v1, v2, w1, w2, scale, k2_bias, v2_bias, inclusive, flags).cast<Tensor>();
    const Args a{w1, w2, scale_of(scale, q), k2_bias, v2_bias, inclusive, flags};
    py::gil_scoped_release nogil;
    if (at::GradMode::is_enabled() &&
        (q.requires_grad() || k1.requires_grad() || k2.requires_grad() || v1.requires_grad() || v2.requires_grad()))
        return Attention::apply(q, k1, k2, v1, v2, a);
    return run_forward(q, k1, k2, v1, v2, a).first;
}

std::pair<Tensor, Tensor> forward(const Tensor& q, const Tensor& k1, const Tensor& k2, const Tensor& v1, const Tensor& v2, int64_t w1, int64_t w2,
                                  std::optional<double> scale, double k2_bias, double v2_bias, bool inclusive, unsigned flags) {
    if (!inputs_ok(q, k1, k2, v1, v2)) refuse_inputs(q, k1, k2, v1, v2);
    py::gil_scoped_release nogil;
    at::AutoDispatchBelowADInplaceOrView below;
    return run_forward(q, k1, k2, v1, v2, Args{w1, w2, scale_of(scale, q), k2_bias, v2_bias, inclusive, flags});
}

py::tuple backward(const Tensor& q, const Tensor& k1, const Tensor& k2, const Tensor& v1, const Tensor& v2, py::object out_o, py::object lse_o,
                   py::object dout_o, int64_t w1, int64_t w2, std::optional<double> scale, double k2_bias, double v2_bias, unsigned needs,
                   bool inclusive, unsigned flags) {
    if (!inputs_ok(q, k1, k2, v1, v2)) refuse_inputs(q, k1, k2, v1, v2);
    auto tensor = [](const py::object& o) { return THPVariable_Check(o.ptr()) ? THPVariable_Unpack(o.ptr()) : Tensor(); };
    const Tensor out = tensor(out_o), lse = tensor(lse_o), dout = tensor(dout_o);
    if (!saved_ok(q, out, lse, dout)) {
        py::handle checks{check_saved_py};
        checks(q, out_o, lse_o, dout_o);
        throw std::invalid_argument("out, lse and dout must be what the forward of these inputs returned and a gradient of its shape");
    }
    std::array<Tensor, 5> g;
    {
        py::gil_scoped_release nogil;
        at::AutoDispatchBelowADInplaceOrView below;
        g = run_backward(q, k1, k2, v1, v2, out, lse, dout, needs, Args{w1, w2, scale_of(scale, q), k2_bias, v2_bias, inclusive, flags});
    }
    py::tuple r(5);
    for (int i = 0; i < 5; ++i) r[i] = g[i].defined() ? py::cast(g[i]) : py::none();
    return r;
}

}  // namespace

PYBIND11_MODULE(_sa2_torch, m) {
    m.doc() = "Native host path of the 2-simplicial attention operator";
    m.def("bind", [](uintptr_t fwd, uintptr_t fwd_ws, uintptr_t bwd, uintptr_t ws, uintptr_t err, py::object check_inputs, py::object check_saved, py::object error,
                     py::object general) {
        fwd_fn = (decltype(fwd_fn))fwd;
        fwd_ws_fn = (decltype(fwd_ws_fn))fwd_ws;
        bwd_fn = (decltype(bwd_fn))bwd;
        ws_fn = (decltype(ws_fn))ws;
        err_fn = (decltype(err_fn))err;
        check_inputs_py = check_inputs.release().ptr();         // kept for the process
        check_saved_py = check_saved.release().ptr();
        general_py = general.release().ptr();
        static PyObject* error_class = nullptr;
        error_class = error.release().ptr();
        py::register_exception_translator([](std::exception_ptr p) {
            try {
                if (p) std::rethrow_exception(p);
            } catch (const Status& s) {
                py::handle make{error_class};
                const py::object e = make(s.code, err_fn(s.code));
                PyErr_SetObject(error_class, e.ptr());
            }
        });
    });
    m.def("attention", &attention);
    m.def("forward", &forward);
    m.def("backward", &backward);
}
