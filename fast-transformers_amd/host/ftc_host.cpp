// Python binding of the C ABI (include/ftc_causal_product.h): the entry points of
// fast_transformers_amd.causal_product take their tensors here.
//
// What bounds a small or ordinary call is the host: with the tensors described through ctypes a
// training step took the host 159 us (one chain of 64 positions), where the two kernels of N=10,
// H=8, L=1000, E=M=64 take 68.  Here a call checks its tensors, describes them on the stack, looks
// its workspace up and launches: 4.3 to 5.2 us per call where ctypes took 16.6 to 21.7; nothing of a
// tensor is kept.
//
// The workspaces stay Python's (causal_product.__init__: one per device and stream, in a dict that
// check_workspaces() walks); they are found here through that dict, and Python is called when
// one has to be made or grown, when an error word has come back and, every ten milliseconds at
// most, to send for the next one.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/csrc/utils/pybind.h>

#include <pybind11/stl.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/SavedTensorHooks.h>
#include <ATen/record_function.h>
#include <ATen/core/grad_mode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdlib>
#include <map>
#include <mutex>
#include <string>
#include <tuple>
#include <vector>

#include "ftc_causal_product.h"

namespace {

namespace py = pybind11;
using at::Tensor;
using OptTensor = std::optional<Tensor>;

[[noreturn]] void error(const std::string &what) { throw std::runtime_error(what); }

void check(int64_t rc, const char *what) {
    if (rc < 0)
        error(std::string(what) + " failed (status " + std::to_string(rc) + "): " + ftc_last_error());
}

// A call into the library without Python's lock: a launch may block (a full queue), and other
// threads go on meanwhile.  `turn`: held during the call, by one thread at a time.
template <class F>
auto native(F f, std::mutex *turn = nullptr) {
    const py::gil_scoped_release unlocked;
    std::unique_lock<std::mutex> held;
    if (turn) held = std::unique_lock<std::mutex>(*turn);
    return f();
}

int32_t dtype_code(const Tensor &t) {
    if (t.scalar_type() == at::kFloat) return FTC_F32;
    if (t.scalar_type() == at::kBFloat16) return FTC_BF16;
    error("causal_dot_product: expected float32 or bfloat16 tensors, got " +
          py::str(py::cast(t.scalar_type())).cast<std::string>());
}

ftc_tensor4 describe(const Tensor &t) {
    ftc_tensor4 d;
    d.ptr = t.numel() == 0 ? nullptr : t.data_ptr();
    d.dtype = dtype_code(t);
    for (int i = 0; i < 4; i++) d.size[i] = t.size(i), d.stride[i] = t.stride(i);
    return d;
}

// The kernels take any N/H/L strides but need unit stride in the last dimension; rows that
// overlap (an expanded L dimension) would take the slow general path.  Zero strides over N or H
// (one sequence shared by chains) are read as they are.
Tensor prepare(const Tensor &t, const char *name) {
    if (t.dim() != 4)
        error(std::string("causal_dot_product: ") + name + " must be 4-dimensional (N, H, L, X), got " +
              std::to_string(t.dim()) + "-d");
    if (!t.is_cuda())
        error(std::string("causal_dot_product: ") + name + " is on " + t.device().str() +
              ", expected a GPU tensor");
    if ((t.size(3) > 1 && t.stride(3) != 1) || (t.size(2) > 1 && t.stride(2) < t.size(3)))
        return t.contiguous();
    return t;
}
const Tensor &check_out(const Tensor &t, const char *name) {
    if (t.dim() != 4 || !t.is_cuda())
        error(std::string("causal_dot_product: ") + name + " must be a 4-dimensional GPU tensor");
    if (t.size(3) > 1 && t.stride(3) != 1)
        error(std::string("causal_dot_product: output ") + name + " must be contiguous in its last dimension");
    return t;
}

// ---- workspaces ----
// (kept for the life of the process: never released, Python may be gone by then)
struct PythonSide {
    py::dict workspaces, probes;
    py::function make_workspace, watch, probe, check_all;
};
PythonSide *g_python = nullptr;

void setup(py::dict workspaces, py::dict probes, py::function make_workspace, py::function watch,
           py::function probe, py::function check_all) {
    g_python = new PythonSide{workspaces, probes, make_workspace, watch, probe, check_all};
}

// Whether the last probe of a workspace has brought back an error word.  (Pinned memory that the
// copy behind an earlier call fills; zero until it arrives.)
bool failed(const py::object &key) {
    PyObject *probe = PyDict_GetItem(g_python->probes.ptr(), key.ptr());  // (borrowed)
    if (!probe) return false;
    const Tensor &word = THPVariable_Unpack(PyList_GetItem(probe, 0));
    return *(const volatile int32_t *)word.const_data_ptr() != 0;
}

// bytes asked for by (query, sizes, dtype): sizes repeat call after call (under Python's lock)
using Query = int64_t (*)(int64_t, int64_t, int64_t, int64_t, int64_t, int32_t);
using SizeKey = std::tuple<Query, int64_t, int64_t, int64_t, int64_t, int64_t, int32_t>;
std::map<SizeKey, int64_t> g_sizes;
void forget_sizes() { g_sizes.clear(); }
int64_t workspace_bytes(Query query, const char *name, int64_t N, int64_t H, int64_t L, int64_t E,
                        int64_t M, int32_t code) {
    const SizeKey key{query, N, H, L, E, M, code};
    const auto it = g_sizes.find(key);
    if (it != g_sizes.end()) return it->second;
    const int64_t bytes = native([&] { return query(N, H, L, E, M, code); });
    check(bytes, name);
    if (g_sizes.size() >= 4096) g_sizes.clear();
    g_sizes[key] = bytes;
    return bytes;
}

// One call's stream and workspace, and the watch on the workspace's error word around it.
struct Call {
    c10::DeviceGuard guard;
    hipStream_t stream;
    Tensor workspace;
    void *ws = nullptr;
    size_t ws_bytes = 0;
    py::object key;
    bool due = false;
    // A call's launches pass data on through the workspace, which all calls on a stream share:
    // another thread's must not come between them.
    std::mutex *turn = nullptr;

    Call(const Tensor &q, int64_t bytes) : guard(q.device()) {
        stream = c10::hip::getCurrentHIPStream(q.device().index()).stream();
        if (bytes <= 0) return;
        key = py::make_tuple((int)q.device().index(), (int64_t)(intptr_t)stream);
        PyObject *found = PyDict_GetItem(g_python->workspaces.ptr(), key.ptr());  // (borrowed)
        if (found) workspace = THPVariable_Unpack(found);
        if (!found || workspace.numel() < bytes)
            workspace = g_python->make_workspace(bytes, key).cast<Tensor>();
        if (failed(key)) g_python->check_all();
        ws = workspace.data_ptr(), ws_bytes = (size_t)workspace.numel();
        using clock = std::chrono::steady_clock;
        struct Shared {
            clock::time_point then;
            std::mutex turn;
        };
        static std::map<std::pair<int, intptr_t>, Shared> shared;  // (under Python's lock)
        Shared &mine = shared[{(int)q.device().index(), (intptr_t)stream}];
        turn = &mine.turn;
        const auto now = clock::now();
        due = now - mine.then >= std::chrono::milliseconds(10);
        if (due) {
            mine.then = now;
            g_python->watch(key, workspace);
        }
    }
    void done() {
        const char *env = getenv("FTC_CHECK");
        if (env && *env && std::string(env) != "0")
            g_python->check_all();
        else if (due)
            g_python->probe(key, workspace);
    }
};

// ---- entry points ----
void forward(const Tensor &queries, const Tensor &keys, const Tensor &values, const Tensor &product) {
    const at::NoGradGuard no_grad;
    const Tensor q = prepare(queries, "queries"), k = prepare(keys, "keys"), v = prepare(values, "values");
    const ftc_tensor4 dq = describe(q), dk = describe(k), dv = describe(v),
                      dout = describe(check_out(product, "product"));
    Call call(q, workspace_bytes(ftc_causal_dot_product_workspace_bytes,
                                 "ftc_causal_dot_product_workspace_bytes", q.size(0), q.size(1), q.size(2),
                                 q.size(3), v.size(3), dq.dtype));
    const int rc = native(
        [&] { return ftc_causal_dot_product(&dq, &dk, &dv, &dout, call.ws, call.ws_bytes, call.stream); }, call.turn);
    check(rc, "ftc_causal_dot_product");
    call.done();
}

std::tuple<Tensor, OptTensor> product_with_state(const Tensor &queries, const Tensor &keys,
                                                 const Tensor &values, const OptTensor &initial_state,
                                                 bool return_state) {
    const at::NoGradGuard no_grad;
    const Tensor q = prepare(queries, "queries"), k = prepare(keys, "keys"), v = prepare(values, "values");
    const int64_t N = q.size(0), H = q.size(1), L = q.size(2), E = q.size(3), M = v.size(3);
    Tensor s0;
    if (initial_state) {
        s0 = prepare(*initial_state, "initial_state");
        if (s0.scalar_type() != at::kFloat || s0.sizes() != at::IntArrayRef({N, H, E, M}))
            error("causal_dot_product_with_state: initial_state must be a float32 tensor of shape "
                  "(N, H, E, M)");
    }
    const auto fp32 = q.options().dtype(at::kFloat);
    const Tensor out = at::empty({N, H, L, M}, fp32);
    OptTensor s1;
    if (return_state) s1 = at::empty({N, H, E, M}, fp32);
    const ftc_tensor4 dq = describe(q), dk = describe(k), dv = describe(v), dout = describe(out);
    ftc_tensor4 d0, d1;
    if (s0.defined()) d0 = describe(s0);
    if (s1) d1 = describe(*s1);
    Call call(q, workspace_bytes(ftc_causal_dot_product_workspace_bytes,
                                 "ftc_causal_dot_product_workspace_bytes", N, H, L, E, M, dq.dtype));
    const int rc = native([&] {
        return ftc_causal_dot_product_state(&dq, &dk, &dv, s0.defined() ? &d0 : nullptr, &dout,
                                            s1 ? &d1 : nullptr, call.ws, call.ws_bytes, call.stream);
    }, call.turn);
    check(rc, "ftc_causal_dot_product_state");
    call.done();
    return {out, s1};
}

// up to nine optional descriptors and what they describe
struct Out {
    ftc_tensor4 d;
    const ftc_tensor4 *p = nullptr;
    Out(const OptTensor &t, const char *name) {
        if (t) d = describe(check_out(*t, name)), p = &d;
    }
};

void backward(const Tensor &queries, const Tensor &keys, const Tensor &values, const Tensor &grad_out,
              const OptTensor &grad_queries, const OptTensor &grad_keys, const OptTensor &grad_values) {
    const at::NoGradGuard no_grad;
    const Tensor q = prepare(queries, "queries"), k = prepare(keys, "keys"), v = prepare(values, "values");
    Tensor g = prepare(grad_out, "grad_out");
    if (g.scalar_type() != at::kFloat) g = g.to(at::kFloat);
    const ftc_tensor4 dq = describe(q), dk = describe(k), dv = describe(v), dg = describe(g);
    const Out gq(grad_queries, "grad_queries"), gk(grad_keys, "grad_keys"), gv(grad_values, "grad_values");
    Call call(q, workspace_bytes(ftc_causal_dot_backward_workspace_bytes,
                                 "ftc_causal_dot_backward_workspace_bytes", q.size(0), q.size(1),
                                 q.size(2), q.size(3), v.size(3), dq.dtype));
    const int rc = native([&] {
        return ftc_causal_dot_backward(&dq, &dk, &dv, &dg, gq.p, gk.p, gv.p, call.ws, call.ws_bytes,
                                       call.stream);
    }, call.turn);
    check(rc, "ftc_causal_dot_backward");
    call.done();
}

const int64_t *lengths_ptr(const OptTensor &lengths, const Tensor &q) {
    if (!lengths) return nullptr;
    if (lengths->scalar_type() != at::kLong || lengths->device() != q.device() || lengths->dim() != 1 ||
        lengths->size(0) != q.size(0) || !lengths->is_contiguous())
        error("causal_linear_attention: key_lengths must be a contiguous int64 tensor of N values on "
              "the device of the queries");
    return lengths->const_data_ptr<int64_t>();
}

// (`wide`: rows of 128 values too)
void fused_attention(const Tensor &queries, const Tensor &keys, const Tensor &values, const OptTensor &key_lengths,
                     double eps, const Tensor &out, const OptTensor &denominators, bool wide) {
    const at::NoGradGuard no_grad;
    const Tensor q = prepare(queries, "queries"), k = prepare(keys, "keys"), v = prepare(values, "values");
    const int64_t *lengths = lengths_ptr(key_lengths, q);
    const ftc_tensor4 dq = describe(q), dk = describe(k), dv = describe(v),
                      dout = describe(check_out(out, "out"));
    ftc_tensor4 dden;
    if (denominators) dden = describe(denominators->unsqueeze(3));
    Call call(q, workspace_bytes(wide ? ftc_causal_linear_attention_wide_workspace_bytes
                                      : ftc_causal_linear_attention_workspace_bytes,
                                 "ftc_causal_linear_attention_workspace_bytes", q.size(0), q.size(1),
                                 q.size(2), q.size(3), v.size(3), dq.dtype));
    const auto run = wide ? ftc_causal_linear_attention_wide_forward : ftc_causal_linear_attention_forward;
    const int rc = native([&] {
        return run(&dq, &dk, &dv, lengths, (float)eps, &dout, denominators ? &dden : nullptr, call.ws, call.ws_bytes,
                   call.stream);
    }, call.turn);
    check(rc, "ftc_causal_linear_attention_forward");
    call.done();
}
void attention(const Tensor &queries, const Tensor &keys, const Tensor &values, const OptTensor &key_lengths,
               double eps, const Tensor &out, const OptTensor &denominators) {
    fused_attention(queries, keys, values, key_lengths, eps, out, denominators, false);
}

void fused_attention_backward(const Tensor &queries, const Tensor &keys, const Tensor &values,
                              const OptTensor &key_lengths, const Tensor &out, const Tensor &denominators,
                              const Tensor &grad_out, const OptTensor &grad_queries, const OptTensor &grad_keys,
                              const OptTensor &grad_values, bool wide) {
    const at::NoGradGuard no_grad;
    const Tensor q = prepare(queries, "queries"), k = prepare(keys, "keys"), v = prepare(values, "values"),
                 o = prepare(out, "out"), g = prepare(grad_out, "grad_out");
    const int64_t *lengths = lengths_ptr(key_lengths, q);
    const ftc_tensor4 dq = describe(q), dk = describe(k), dv = describe(v), dout = describe(o),
                      dden = describe(denominators.unsqueeze(3)), dg = describe(g);
    const Out gq(grad_queries, "grad_queries"), gk(grad_keys, "grad_keys"), gv(grad_values, "grad_values");
    Call call(q, workspace_bytes(wide ? ftc_causal_linear_attention_wide_backward_workspace_bytes
                                      : ftc_causal_linear_attention_backward_workspace_bytes,
                                 "ftc_causal_linear_attention_backward_workspace_bytes", q.size(0),
                                 q.size(1), q.size(2), q.size(3), v.size(3), dq.dtype));
    const auto run = wide ? ftc_causal_linear_attention_wide_backward : ftc_causal_linear_attention_backward;
    const int rc = native([&] {
        return run(&dq, &dk, &dv, lengths, &dout, &dden, &dg, gq.p, gk.p, gv.p, call.ws, call.ws_bytes, call.stream);
    }, call.turn);
    check(rc, "ftc_causal_linear_attention_backward");
    call.done();
}
void attention_backward(const Tensor &queries, const Tensor &keys, const Tensor &values,
                        const OptTensor &key_lengths, const Tensor &out, const Tensor &denominators,
                        const Tensor &grad_out, const OptTensor &grad_queries, const OptTensor &grad_keys,
                        const OptTensor &grad_values) {
    fused_attention_backward(queries, keys, values, key_lengths, out, denominators, grad_out, grad_queries, grad_keys,
                             grad_values, false);
}

// ---- the differentiable entry points ----
// A training step of a few short sequences is bound by the host: 80 us, of which the GPU works 20.
// As torch.autograd.Function in Python the two directions cost their share of the interpreter, on
// the engine's thread too; here they are functions of the C++ engine.  Measured (a step as
// autograd.grad): causal_dot_product, 3 x 8 chains, L=529 79 -> 63 us (what is left is mostly the two
// changes of thread), N=10, H=8, L=1000 76.5 -> 69; the attention module, 3 x 4 chains, L=189
// 131 -> 83.
//
// Only plain calls are taken: exact tensors or parameters on the GPU, rows of a type that the kernels
// take, and nothing that watches or transforms operations (function and dispatch modes, functorch,
// forward-mode gradients, saved-tensor hooks, tracing).  Everything else is answered with None, and
// the caller goes on with the Python function, which treats such calls as it always has.
// (bit by bit: a difference of key sets keeps the backends' bits)
bool only(c10::DispatchKeySet keys, c10::DispatchKeySet allowed) {
    return (keys.raw_repr() & ~allowed.raw_repr()) == 0;
}
const Tensor *plain(py::handle h) {
    if (!THPVariable_CheckExact(h.ptr())) return nullptr;
    const Tensor &t = THPVariable_Unpack(h.ptr());
    using K = c10::DispatchKey;
    constexpr c10::DispatchKeySet usual =
        c10::DispatchKeySet({K::CUDA, K::AutogradCUDA, K::ADInplaceOrView, K::AutocastCUDA});
    const bool ok = t.defined() && t.is_cuda() && t.dim() == 4 && t.layout() == at::kStrided && !t.is_inference() &&
                    only(t.key_set(), usual) && !t._fw_grad(0).defined();
    return ok ? &t : nullptr;
}
bool nothing_watches() {
    const auto tls = c10::impl::tls_local_dispatch_key_set();
    return only(tls.included_, c10::default_included_set | c10::autocast_dispatch_keyset) &&
           only(tls.excluded_, c10::default_excluded_set) && !c10::impl::TorchDispatchModeTLS::any_modes_set() &&
           at::impl::PythonTorchFunctionTLS::stack_len() == 0 && !at::SavedTensorDefaultHooks::get_hooks() &&
           !torch::jit::tracer::isTracing() && !c10::InferenceMode::is_enabled();
}
bool differentiated(std::initializer_list<const Tensor *> inputs) {
    if (!at::GradMode::is_enabled()) return false;
    for (const Tensor *t : inputs)
        if (t->requires_grad()) return true;
    return false;
}
// The engine calls back on a thread of its own, without Python's lock, and carries exceptions to the
// thread that waits: one of Python's in the form that it knows to.
template <class F>
void from_engine(F f) {
    const py::gil_scoped_acquire locked;
    try {
        f();
    } catch (py::error_already_set &e) {
        e.restore();
        python_error held;
        held.persist();
        throw held;
    }
}

using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

struct CausalDot : torch::autograd::Function<CausalDot> {
    static Tensor run(const Tensor &q, const Tensor &k, const Tensor &v) {
        // (the kernels overwrite every element)
        const Tensor product = at::empty({q.size(0), q.size(1), q.size(2), v.size(3)}, q.options().dtype(at::kFloat));
        ::forward(q, k, v, product);
        return product;
    }
    static Tensor forward(AutogradContext *ctx, const Tensor &q, const Tensor &k, const Tensor &v) {
        ctx->save_for_backward({q, k, v});
        return run(q, k, v);
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        RECORD_FUNCTION("CausalDotProductBackward", std::vector<c10::IValue>());
        const variable_list saved = ctx->get_saved_variables();
        variable_list out;
        for (const Tensor &t : saved) out.push_back(at::empty_like(t, at::MemoryFormat::Contiguous));
        from_engine([&] { ::backward(saved[0], saved[1], saved[2], grads[0], out[0], out[1], out[2]); });
        return out;
    }
};

// causal_product.CausalDotProduct.apply on plain tensors; None: not such a call
py::object dot(py::handle queries, py::handle keys, py::handle values) {
    const Tensor *q = plain(queries), *k = plain(keys), *v = plain(values);
    if (!q || !k || !v || !nothing_watches()) return py::none();
    // (a profiler's ranges are those of the Python functions)
    RECORD_FUNCTION("CausalDotProduct", std::vector<c10::IValue>({*q, *k, *v}));
    return py::cast(differentiated({q, k, v}) ? CausalDot::apply(*q, *k, *v) : CausalDot::run(*q, *k, *v));
}

Tensor swapped(const Tensor &t) { return t.permute({0, 2, 1, 3}); }

// rows of 128 values
bool wide_rows(const Tensor &q, const Tensor &v) { return q.size(-1) > 64 || v.size(-1) > 64; }
// ... are read where 16-byte loads reach them in chains within 2 GiB (t as the module has it)
bool reads_in_place(const Tensor &t) {
    const int64_t row = std::max(t.stride(1), t.size(2) * t.size(3));
    return (uintptr_t)t.const_data_ptr() % 16 == 0 && t.stride(3) == 1 && t.stride(0) % 4 == 0 &&
           t.stride(1) % 4 == 0 && t.stride(2) % 4 == 0 && t.stride(1) >= t.size(3) && row <= (1 << 16) &&
           (t.size(1) + 64) * row * 4 < 0x7fffffff;
}

// tensors as the attention module has them, (N, L, H, X)
struct CausalAttention : torch::autograd::Function<CausalAttention> {
    static Tensor run(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &lengths, double eps,
                      const OptTensor &denominators) {
        const Tensor out = at::empty({q.size(0), q.size(1), q.size(2), v.size(3)}, q.options());
        ::fused_attention(swapped(q), swapped(k), swapped(v), lengths, eps, swapped(out), denominators, wide_rows(q, v));
        return out;
    }
    static Tensor forward(AutogradContext *ctx, const Tensor &q, const Tensor &k, const Tensor &v,
                          const Tensor &lengths, double eps) {
        RECORD_FUNCTION("CausalLinearAttentionFunction", std::vector<c10::IValue>({q, k, v}));
        const Tensor den = at::empty({q.size(0), q.size(2), q.size(1)}, q.options());
        const Tensor out = run(q, k, v, lengths, eps, den);
        if (wide_rows(q, v)) {
            // The composition does not keep its result, which the caller may then change in place: kept here
            // as an alias that no check refuses, with a tensor that tells such a change (it shares the
            // result's version), after which the backward computes the result again.
            const Tensor version = at::empty({0});
            torch::autograd::impl::set_version_counter(version, torch::autograd::impl::version_counter(out));
            ctx->saved_data["version"] = version;
            ctx->saved_data["unchanged"] = (int64_t)out._version();
            // (queries and keys that nothing is derived for: the composition keeps their features, not them)
            auto own = [](const Tensor &t) { return t.requires_grad() ? t : t.clone(); };
            ctx->save_for_backward({own(q), own(k), v, out.variable_data(), den});
        } else {
            ctx->save_for_backward({q, k, v, out, den});
        }
        // (rows of 128: as in the composition, which makes its mask here, the caller may have the lengths back)
        const at::AutoDispatchBelowADInplaceOrView below;  // (a plain copy costs the host half as much)
        ctx->saved_data["lengths"] = wide_rows(q, v) ? at::empty_like(lengths).copy_(lengths) : lengths;
        ctx->saved_data["eps"] = eps;
        return out;
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        RECORD_FUNCTION("CausalLinearAttentionFunctionBackward", std::vector<c10::IValue>());
        const variable_list saved = ctx->get_saved_variables();
        const Tensor lengths = ctx->saved_data["lengths"].toTensor();
        variable_list out(5);
        OptTensor to[3];
        if (wide_rows(saved[0], saved[2]) && at::GradMode::is_enabled()) {
            // (the caller means to differentiate again: the composition's gradients, whose element-wise parts
            // can be)
            from_engine([&] {
                const py::tuple needed = py::make_tuple(ctx->needs_input_grad(0), ctx->needs_input_grad(1),
                                                        ctx->needs_input_grad(2));
                const auto composed = py::module_::import("fast_transformers_amd.attention.causal_linear_attention")
                                          .attr("composed_gradients")(saved[0], saved[1], saved[2], lengths,
                                                                      ctx->saved_data["eps"].toDouble(), grads[0], needed)
                                          .cast<std::vector<OptTensor>>();
                for (int i = 0; i < 3; i++)
                    if (composed[i]) out[i] = *composed[i];
            });
            return out;
        }
        for (int i = 0; i < 3; i++)
            if (ctx->needs_input_grad(i)) out[i] = at::empty_like(saved[i]), to[i] = swapped(out[i]);
        from_engine([&] {
            const bool wide = wide_rows(saved[0], saved[2]);
            Tensor result = saved[3];
            if (wide && (int64_t)ctx->saved_data["version"].toTensor()._version() != ctx->saved_data["unchanged"].toInt())
                result = run(saved[0], saved[1], saved[2], lengths, ctx->saved_data["eps"].toDouble(), std::nullopt);
            const Tensor g = wide && !reads_in_place(grads[0]) ? grads[0].clone(at::MemoryFormat::Contiguous) : grads[0];
            ::fused_attention_backward(swapped(saved[0]), swapped(saved[1]), swapped(saved[2]), lengths,
                                       swapped(result), saved[4], swapped(g), to[0], to[1], to[2], wide);
        });
        return out;
    }
};

// The fused forward of the attention module; None: not a plain call, or sizes without a fused kernel
// (mask_length: how many positions the mask of the lengths has, -1 if unknown)
py::object attention_module(py::handle queries, py::handle keys, py::handle values, py::handle key_lengths,
                            int64_t mask_length, double eps) {
    const Tensor *q = plain(queries), *k = plain(keys), *v = plain(values);
    if (!q || !k || !v || !THPVariable_CheckExact(key_lengths.ptr()) || !nothing_watches()) return py::none();
    const Tensor &lengths = THPVariable_Unpack(key_lengths.ptr());
    auto width = [](int64_t w) { return w == 32 || w == 64 || w == 128; };
    for (const Tensor *t : {q, k, v})
        if (t->scalar_type() != at::kFloat || t->device() != q->device() || t->size(1) != q->size(1)) return py::none();
    if (k->size(3) != q->size(3) || !width(q->size(3)) || !width(v->size(3)) || lengths.device() != q->device() ||
        lengths.scalar_type() != at::kLong || !lengths.is_contiguous() || lengths.requires_grad())
        return py::none();
    if (wide_rows(*q, *v)) {  // (what the composition would broadcast or refuse is left to it)
        if (lengths.dim() != 1 || lengths.size(0) != q->size(0) || mask_length != q->size(1) || std::isnan(eps))
            return py::none();
        for (const Tensor *t : {q, k, v})
            if (!reads_in_place(*t) || t->size(0) != q->size(0) || t->size(2) != q->size(2)) return py::none();
        if (ftc_causal_linear_attention_wide_workspace_bytes(q->size(0), q->size(2), q->size(1), q->size(3), v->size(3),
                                                             FTC_F32) < 0)
            return py::none();
    }
    return py::cast(differentiated({q, k, v}) ? CausalAttention::apply(*q, *k, *v, lengths, eps)
                                              : CausalAttention::run(*q, *k, *v, lengths, eps, std::nullopt));
}

// ---- the encoder's forward, eval mode ----
struct Linear {
    Tensor weight;
    OptTensor bias;
};
struct Norm {
    OptTensor weight, bias;
    double eps;
};
struct Layer {
    Linear query, key, value, out, first, second;
    Norm norm1, norm2;
    double eps;
};

// One weight matrix (or several with the same number of columns, their rows one after the other)
// in pieces, in memory that is handed out from `at` on.
struct Pieces {
    const float *pieces, *scale, *bias, *norm;
    int64_t rows, cols;
    static int64_t floats(std::initializer_list<const Linear *> parts) {
        int64_t n = 0;
        for (const Linear *l : parts) n += l->weight.size(0) * (l->weight.size(1) + 3);
        return n;
    }
    Pieces(std::initializer_list<const Linear *> parts, std::vector<ftc_weight> &list, float *&at) {
        rows = 0, cols = (*parts.begin())->weight.size(1);
        for (const Linear *l : parts) rows += l->weight.size(0);
        float *const p = at, *const s = p + rows * cols, *const b = s + rows, *const n = b + rows;
        at = n + rows;
        pieces = p, scale = s, bias = b, norm = n;
        int64_t row = 0;
        for (const Linear *l : parts) {
            ftc_weight w;
            w.w = l->weight.const_data_ptr<float>();
            w.bias = l->bias ? l->bias->const_data_ptr<float>() : nullptr;
            w.rows = l->weight.size(0), w.cols = cols;
            w.pieces = p + row * cols, w.scale = s + row, w.bias_out = b + row, w.norm = n + row;
            list.push_back(w);
            row += w.rows;
        }
    }
};
// The weights of consecutive layers in pieces, cut in one launch.
struct LayerPieces {
    Pieces in, proj, first, second;
    static int64_t floats(const Layer &l) {
        return Pieces::floats({&l.query, &l.key, &l.value, &l.out, &l.first, &l.second});
    }
    LayerPieces(const Layer &l, std::vector<ftc_weight> &list, float *&at)
        : in({&l.query, &l.key, &l.value}, list, at), proj({&l.out}, list, at), first({&l.first}, list, at),
          second({&l.second}, list, at) {}
};
// How many layers from `from` on have their weights cut at a time.  Few tokens: all of them, up to eight with
// pieces of up to 64 MB, since a launch for each (5 to 9 us, much of it latency) is then a tenth of a layer's time.  With
// more, where the rows of x have twice as many values as a layer's weights, one: the others' pieces
// would be memory that the modules do not need, for 1 % of the time.
// Eight layers, 4 x 338 tokens, d = 512 and feed-forward 512: 652 -> 575 us; four, 2 x 966, d = 128: 317 -> 250.
size_t layers_at_a_time(const std::vector<Layer> &layers, size_t from, int64_t values) {
    int64_t floats = LayerPieces::floats(layers[from]);
    if (values > 2 * floats) return 1;
    size_t n = 1;
    while (n < 8 && from + n < layers.size()) {
        floats += LayerPieces::floats(layers[from + n]);
        if (4 * floats > (int64_t)64 << 20) break;
        n++;
    }
    return n;
}

// A stack of post-norm encoder layers (attention/encoder.py) with causal linear attention, and the
// final norm: every product on the fp16 matrix cores in pieces (csrc/ftc_linear.hip), the norms
// leaving their rows in pieces as well.  `x`: dense (N, L, d).
//
// Memory: rows are kept only as long as they are read, so that the stack needs no more than its
// modules did (five times x where the feed-forward layer has at most 3 d features: twelve with a
// buffer for each of them).  `wide` holds a layer's q, k and v; when the attention has read them, its
// rows in pieces; then the feed-forward rows.  `rows` begins a layer with x in pieces and has the attention's
// rows and either norm's pieces in turn.  `out` has the rows before a norm, to which the next product adds the
// norm of what was there; norms inside the stack leave their pieces and two numbers a row (stats).
Tensor encoder(const Tensor &x, const std::vector<Layer> &layers, const std::optional<Norm> &final_norm,
               int64_t H, int64_t E, int64_t M, const OptTensor &key_lengths) {
    const at::NoGradGuard no_grad;
    const int64_t N = x.size(0), L = x.size(1), d = x.size(2), T = N * L;
    const auto fp32 = x.options();
    const int64_t *lengths = lengths_ptr(key_lengths, x);
    const int64_t width = H * (2 * E + M), most_rows = std::max(d, H * M);
    int64_t most_wide = width;
    for (const Layer &l : layers) most_wide = std::max(most_wide, l.first.weight.size(0));
    const Tensor wide = at::empty({T, most_wide}, fp32), scale_of_rows = at::empty({T}, fp32),
                 scale_of_wide = at::empty({T}, fp32), out = at::empty_like(x);
    const Tensor rows_buffer = at::empty({T, most_rows}, fp32), stats_of_rows = at::empty({T, 2}, fp32);
    float *const qkv = wide.data_ptr<float>(), *const rows = rows_buffer.data_ptr<float>();
    float *const stats = stats_of_rows.data_ptr<float>();
    float *const row_scale = scale_of_rows.data_ptr<float>(), *const wide_scale = scale_of_wide.data_ptr<float>();
    float *const to = out.data_ptr<float>();
    auto view = [&](float *base, int64_t column, int64_t row, int64_t X) {
        ftc_tensor4 v;
        v.ptr = base + column, v.dtype = FTC_F32;
        v.size[0] = N, v.size[1] = H, v.size[2] = L, v.size[3] = X;
        v.stride[0] = L * row, v.stride[1] = X, v.stride[2] = row, v.stride[3] = 1;
        return v;
    };
    const ftc_tensor4 q = view(qkv, 0, width, E), k = view(qkv, H * E, width, E),
                      v = view(qkv, 2 * H * E, width, M);
    Call call(x, workspace_bytes(ftc_causal_linear_attention_workspace_bytes,
                                 "ftc_causal_linear_attention_workspace_bytes", N, H, L, E, M, FTC_F32));
    void *const stream = call.stream;
    auto f = [](const OptTensor &t) { return t ? t->const_data_ptr<float>() : nullptr; };
    // (whoever writes rows of so many values asks first: d, the heads' widths and the feed-forward width are
    // independent of each other)
    auto room = [&](float *base, int64_t columns) {
        const int64_t most = base == qkv ? most_wide : base == rows ? most_rows : d;
        TORCH_CHECK(columns <= most, "rows of ", columns, " values in a buffer for ", most);
        return base;
    };
    // (either the rows themselves or, behind max(., 0), in pieces with a scale)
    auto linear = [&](const float *pieces, const float *pieces_scale, const Pieces &w, const float *residual,
                      float *y, float *relu_pieces, float *relu_scale) {
        check(ftc_linear_split(pieces, pieces_scale, T, w.pieces, w.scale, w.bias, w.norm, w.rows, w.cols, residual,
                               y ? room(y, w.rows) : y, relu_pieces ? room(relu_pieces, w.rows) : relu_pieces,
                               relu_scale, stream),
              "ftc_linear_split");
    };
    auto split = [&](const float *from, int64_t columns, float *pieces, float *pieces_scale) {
        check(ftc_split_rows(from, T, columns, room(pieces, columns), pieces_scale, stream), "ftc_split_rows");
    };
    auto norm = [&](const float *from, const Norm &n, float *y) {
        check(ftc_layer_norm_split(from, f(n.weight), f(n.bias), (float)n.eps, T, d, room(y, d), nullptr, nullptr, stream),
              "ftc_layer_norm_split");
    };
    // the norm of `to` in pieces, and what a product needs to add it to its own rows
    auto norm_of_rows = [&](const Norm &n) {
        check(ftc_layer_norm_stats_split(to, f(n.weight), f(n.bias), (float)n.eps, T, d, stats, room(rows, d), row_scale,
                                         stream),
              "ftc_layer_norm_stats_split");
    };
    auto linear_normed = [&](const Pieces &w, const Norm &n, float *y) {
        check(ftc_linear_split_normed(qkv, wide_scale, T, w.pieces, w.scale, w.bias, w.rows, w.cols, to, stats,
                                      f(n.weight), f(n.bias), room(y, w.rows), stream),
              "ftc_linear_split_normed");
    };
    native([&] {
        split(x.const_data_ptr<float>(), d, rows, row_scale);
        Tensor weights;                  // of layers cut_from, cut_from + 1 ... in pieces
        std::vector<LayerPieces> cut;
        size_t cut_from = 0;
        for (size_t i = 0; i < layers.size(); i++) {
            const Layer &l = layers[i];
            if (i == cut_from + cut.size()) {
                const size_t n = layers_at_a_time(layers, i, T * d);
                int64_t floats = 0;
                for (size_t j = i; j < i + n; j++) floats += LayerPieces::floats(layers[j]);
                cut.clear(), cut_from = i;
                weights = Tensor();  // (given back first)
                weights = at::empty({floats}, fp32);
                float *at = weights.data_ptr<float>();
                std::vector<ftc_weight> list;
                for (size_t j = i; j < i + n; j++) cut.emplace_back(layers[j], list, at);
                check(ftc_split_weights(list.data(), (int32_t)list.size(), stream), "ftc_split_weights");
            }
            const LayerPieces &w = cut[i - cut_from];
            linear(rows, row_scale, w.in, nullptr, qkv, nullptr, nullptr);
            const ftc_tensor4 o = view(room(rows, H * M), 0, H * M, M);
            check(ftc_causal_linear_attention_forward(&q, &k, &v, lengths, (float)l.eps, &o, nullptr, call.ws,
                                                      call.ws_bytes, stream),
                  "ftc_causal_linear_attention_forward");
            split(rows, H * M, qkv, wide_scale);
            if (i == 0)
                linear(qkv, wide_scale, w.proj, x.const_data_ptr<float>(), to, nullptr, nullptr);
            else
                linear_normed(w.proj, layers[i - 1].norm2, to);
            norm_of_rows(l.norm1);
            linear(rows, row_scale, w.first, nullptr, nullptr, qkv, wide_scale);
            if (i + 1 < layers.size()) {
                linear_normed(w.second, l.norm1, to);
                norm_of_rows(l.norm2);
            } else {
                // (`wide` need not have room for rows of d values; the other two always do)
                linear_normed(w.second, l.norm1, final_norm ? to : rows);
                norm(final_norm ? to : rows, l.norm2, final_norm ? rows : to);
                if (final_norm) norm(rows, *final_norm, to);
            }
        }
    }, call.turn);
    call.done();
    return out;
}

}  // namespace

PYBIND11_MODULE(_ftc_host, m) {
    m.def("setup", &setup);
    m.def("forget_sizes", &forget_sizes);
    m.def("forward", &forward);
    m.def("product_with_state", &product_with_state);
    m.def("backward", &backward);
    m.def("attention", &attention);
    m.def("attention_backward", &attention_backward);
    m.def("dot", &dot);
    m.def("attention_module", &attention_module);
    py::class_<Linear>(m, "Linear").def(py::init<Tensor, OptTensor>());
    py::class_<Norm>(m, "Norm").def(py::init<OptTensor, OptTensor, double>());
    py::class_<Layer>(m, "Layer").def(
        py::init<Linear, Linear, Linear, Linear, Linear, Linear, Norm, Norm, double>());
    m.def("encoder", &encoder);
}
