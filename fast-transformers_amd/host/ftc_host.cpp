// Python binding of the C ABI (include/ftc_causal_product.h): the entry points of
// fast_transformers_amd.causal_product take their tensors here.
//
// What bounds a small or ordinary call is the host: with the tensors described through ctypes a
// forward + backward pass of N=10, H=8, L=1000, E=M=64 took the host 165 us where its two kernels
// take 68.  Here a call checks its tensors, describes them on the stack, looks its workspace up
// and launches, in about a microsecond and a half; nothing of a tensor is kept.
//
// The workspaces stay Python's (causal_product.__init__: one per device and stream, in a dict that
// check_workspaces() walks); they are found here through that dict, and Python is called when
// one has to be made or grown and, every ten milliseconds at most, to look after its error word.
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>

#include <ATen/ATen.h>
#include <ATen/core/grad_mode.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include <chrono>
#include <cstdlib>
#include <map>
#include <string>
#include <tuple>

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

int32_t dtype_code(const Tensor &t) {
    if (t.scalar_type() == at::kFloat) return FTC_F32;
    if (t.scalar_type() == at::kBFloat16) return FTC_BF16;
    error(std::string("causal_dot_product: expected float32 or bfloat16 tensors, got torch.") +
          at::toString(t.scalar_type()));
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
    py::dict workspaces;
    py::function make_workspace, watch, probe, check_all;
};
PythonSide *g_python = nullptr;

void setup(py::dict workspaces, py::function make_workspace, py::function watch, py::function probe,
           py::function check_all) {
    g_python = new PythonSide{workspaces, make_workspace, watch, probe, check_all};
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
    const int64_t bytes = query(N, H, L, E, M, code);
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

    Call(const Tensor &q, int64_t bytes) : guard(q.device()) {
        stream = c10::hip::getCurrentHIPStream(q.device().index()).stream();
        if (bytes <= 0) return;
        key = py::make_tuple((int)q.device().index(), (int64_t)(intptr_t)stream);
        PyObject *found = PyDict_GetItem(g_python->workspaces.ptr(), key.ptr());  // (borrowed)
        if (found) workspace = THPVariable_Unpack(found);
        if (!found || workspace.numel() < bytes)
            workspace = g_python->make_workspace(bytes, key).cast<Tensor>();
        ws = workspace.data_ptr(), ws_bytes = (size_t)workspace.numel();
        using clock = std::chrono::steady_clock;
        static std::map<std::pair<int, intptr_t>, clock::time_point> last;  // (under Python's lock)
        auto &then = last[{(int)q.device().index(), (intptr_t)stream}];
        const auto now = clock::now();
        due = now - then >= std::chrono::milliseconds(10);
        if (due) {
            then = now;
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
    check(ftc_causal_dot_product(&dq, &dk, &dv, &dout, call.ws, call.ws_bytes, call.stream),
          "ftc_causal_dot_product");
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
    check(ftc_causal_dot_product_state(&dq, &dk, &dv, s0.defined() ? &d0 : nullptr, &dout,
                                       s1 ? &d1 : nullptr, call.ws, call.ws_bytes, call.stream),
          "ftc_causal_dot_product_state");
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
    check(ftc_causal_dot_backward(&dq, &dk, &dv, &dg, gq.p, gk.p, gv.p, call.ws, call.ws_bytes, call.stream),
          "ftc_causal_dot_backward");
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

void attention(const Tensor &queries, const Tensor &keys, const Tensor &values, const OptTensor &key_lengths,
               double eps, const Tensor &out, const OptTensor &denominators) {
    const at::NoGradGuard no_grad;
    const Tensor q = prepare(queries, "queries"), k = prepare(keys, "keys"), v = prepare(values, "values");
    const int64_t *lengths = lengths_ptr(key_lengths, q);
    const ftc_tensor4 dq = describe(q), dk = describe(k), dv = describe(v),
                      dout = describe(check_out(out, "out"));
    ftc_tensor4 dden;
    if (denominators) dden = describe(denominators->unsqueeze(3));
    Call call(q, workspace_bytes(ftc_causal_linear_attention_workspace_bytes,
                                 "ftc_causal_linear_attention_workspace_bytes", q.size(0), q.size(1),
                                 q.size(2), q.size(3), v.size(3), dq.dtype));
    check(ftc_causal_linear_attention_forward(&dq, &dk, &dv, lengths, (float)eps, &dout,
                                              denominators ? &dden : nullptr, call.ws, call.ws_bytes,
                                              call.stream),
          "ftc_causal_linear_attention_forward");
    call.done();
}

void attention_backward(const Tensor &queries, const Tensor &keys, const Tensor &values,
                        const OptTensor &key_lengths, const Tensor &out, const Tensor &denominators,
                        const Tensor &grad_out, const OptTensor &grad_queries, const OptTensor &grad_keys,
                        const OptTensor &grad_values) {
    const at::NoGradGuard no_grad;
    const Tensor q = prepare(queries, "queries"), k = prepare(keys, "keys"), v = prepare(values, "values"),
                 o = prepare(out, "out"), g = prepare(grad_out, "grad_out");
    const int64_t *lengths = lengths_ptr(key_lengths, q);
    const ftc_tensor4 dq = describe(q), dk = describe(k), dv = describe(v), dout = describe(o),
                      dden = describe(denominators.unsqueeze(3)), dg = describe(g);
    const Out gq(grad_queries, "grad_queries"), gk(grad_keys, "grad_keys"), gv(grad_values, "grad_values");
    Call call(q, workspace_bytes(ftc_causal_linear_attention_backward_workspace_bytes,
                                 "ftc_causal_linear_attention_backward_workspace_bytes", q.size(0),
                                 q.size(1), q.size(2), q.size(3), v.size(3), dq.dtype));
    check(ftc_causal_linear_attention_backward(&dq, &dk, &dv, lengths, &dout, &dden, &dg, gq.p, gk.p, gv.p,
                                               call.ws, call.ws_bytes, call.stream),
          "ftc_causal_linear_attention_backward");
    call.done();
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
}
