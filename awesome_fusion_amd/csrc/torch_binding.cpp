// The PyTorch side of the library in native code: the operators torch.ops.awesome_fusion.bfaintb_gemm[_prepacked], the
// linear layer's forward pass as one call, and the launch call behind gemm.py's gemm and gemm_prepacked.
//
// What bounds it: the small products take 5 - 10 us on the GPU, and the same path in Python (a custom operator's wrapper,
// the argument checks, the workspace look-up, two ctypes calls) took 21 - 26 us of host time per call, so every call
// below some 25 us was bound by the host.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/library.h>

#include <algorithm>
#include <atomic>
#include <list>
#include <mutex>
#include <optional>
#include <unordered_map>

#include "../../include/bfaintb_gemm.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;

// ---- split-K workspaces: one per (device, stream).  Calls ordered on a stream may share one, calls on different streams
//      may overlap and must not.  A workspace grows to at least twice its size, and the kMaxWorkspaces most recently used
//      ones are kept.  What a captured graph uses stays until the graph is gone, whatever becomes of it here (a replay does
//      not come through here): the graph owns an object whose end says so.
constexpr size_t kMaxWorkspaces = 64;
constexpr int64_t kFirstWorkspaceBytes = 4 << 20;

// The workspaces of one capture, held until every graph made from it is gone.
struct GraphHold {
    unsigned long long capture;
    std::vector<Tensor> held;
    std::atomic<bool> gone{false};
};
struct WorkspaceKey {
    int device;
    hipStream_t stream;
    bool operator==(const WorkspaceKey& o) const { return device == o.device && stream == o.stream; }
};
struct WorkspaceKeyHash {
    size_t operator()(const WorkspaceKey& k) const { return reinterpret_cast<size_t>(k.stream) / 64u * 31u + (size_t)k.device; }
};
class WorkspacePool {
    std::mutex mutex_;
    struct Workspace {
        Tensor memory;
        std::list<WorkspaceKey>::iterator place;  // in recent_
    };
    std::list<WorkspaceKey> recent_;  // most recently used first
    std::unordered_map<WorkspaceKey, Workspace, WorkspaceKeyHash> pool_;
    std::vector<GraphHold*> graphs_;

    // (called by the runtime, on a thread and under locks of its own, once the last graph is destroyed and has run: the rest is done
    // by drop_gone)
    static void graph_gone(void* hold) { static_cast<GraphHold*>(hold)->gone.store(true, std::memory_order_release); }

    void drop_gone()
    {
        const auto keep = std::partition(graphs_.begin(), graphs_.end(), [](const GraphHold* h) { return !h->gone.load(std::memory_order_acquire); });
        std::for_each(keep, graphs_.end(), [](GraphHold* h) { delete h; });
        graphs_.erase(keep, graphs_.end());
    }

    void hold_for_graph(const Tensor& memory, hipStream_t stream)
    {
        hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
        unsigned long long capture = 0;
        hipGraph_t graph = nullptr;
        const bool known = hipStreamGetCaptureInfo_v2(stream, &status, &capture, &graph, nullptr, nullptr) == hipSuccess && status == hipStreamCaptureStatusActive;
        if (!known) capture = 0;
        auto it = std::find_if(graphs_.begin(), graphs_.end(), [&](const GraphHold* h) { return h->capture == capture; });
        if (it == graphs_.end()) {
            drop_gone();
            graphs_.push_back(new GraphHold{capture, {}});
            it = graphs_.end() - 1;
            hipUserObject_t object;
            const bool owned = known && hipUserObjectCreate(&object, *it, graph_gone, 1, hipUserObjectNoDestructorSync) == hipSuccess &&
                               hipGraphRetainUserObject(graph, object, 1, hipGraphUserObjectMove) == hipSuccess;
            if (!owned) (void)hipGetLastError();  // (nothing will say when the graph is gone: held for good)
        }
        for (const Tensor& t : (*it)->held)
            if (t.is_same(memory)) return;
        (*it)->held.push_back(memory);
    }

public:
    Tensor get(int64_t bytes, const Tensor& like, hipStream_t stream)
    {
        const WorkspaceKey key{like.device().index(), stream};
        hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(stream, &status) != hipSuccess) (void)hipGetLastError();
        const bool capturing = status != hipStreamCaptureStatusNone;
        std::lock_guard<std::mutex> lock(mutex_);
        auto it = pool_.find(key);
        if (it != pool_.end()) recent_.splice(recent_.begin(), recent_, it->second.place);
        if (it != pool_.end() && it->second.memory.numel() >= bytes) {
            if (capturing) hold_for_graph(it->second.memory, stream);
            return it->second.memory;
        }
        int64_t size = std::max(bytes, kFirstWorkspaceBytes);
        if (it != pool_.end() && !capturing) size = std::max(size, 2 * it->second.memory.numel());
        Tensor fresh = at::empty({size}, like.options().dtype(at::kByte));
        const int rc = bfaintb_workspace_init(fresh.data_ptr(), (size_t)size, stream);
        TORCH_CHECK(rc == 0, "bfaintb_workspace_init failed: [", rc, "] ", bfaintb_error_string(rc));
        // (made under capture: the graph's own, filled by the graph's own first node; not for calls outside it)
        if (capturing) return fresh;
        drop_gone();
        if (it != pool_.end()) {
            it->second.memory = fresh;
            return fresh;
        }
        while (pool_.size() >= kMaxWorkspaces) {
            pool_.erase(recent_.back());
            recent_.pop_back();
        }
        recent_.push_front(key);
        pool_.emplace(key, Workspace{fresh, recent_.begin()});
        return fresh;
    }
    void clear()
    {
        std::lock_guard<std::mutex> lock(mutex_);
        pool_.clear();
        recent_.clear();
        drop_gone();
    }
};
WorkspacePool& workspaces()
{
    static WorkspacePool* pool = new WorkspacePool;  // (never destroyed: the HIP runtime may be gone by then)
    return *pool;
}

// ---- errors of the library as the exception the Python package defines (a RuntimeError with a .code)
PyObject* g_error_class = nullptr;

[[noreturn]] void raise_library_error(int rc, const char* what)
{
    if (g_error_class == nullptr) TORCH_CHECK(false, what, " failed: [", rc, "] ", bfaintb_error_string(rc));
    PyGILState_STATE gil = PyGILState_Ensure();
    PyObject* e = PyObject_CallFunction(g_error_class, "is", rc, what);
    if (e != nullptr) {
        PyErr_SetObject(g_error_class, e);
        Py_DECREF(e);
    }
    python_error err;
    err.persist();
    PyGILState_Release(gil);
    throw err;
}

struct Shape {
    int64_t m, n, k, out_n;
};

int64_t out_columns(int64_t n, int64_t activation)
{
    TORCH_CHECK_VALUE(activation == 0 || activation == 1, "bfaintb_gemm: activation must be 0 (none) or 1 (SiLU gate)");
    return activation == 1 ? n / 2 : n;
}

Shape check(const Tensor& a, const Tensor& w, const Tensor& scale, int64_t bits, int64_t group, const OptTensor& bias, const OptTensor& residual,
            int64_t activation, bool packed)
{
    const char* name = packed ? "bfaintb_gemm_prepacked" : "bfaintb_gemm";
    TORCH_CHECK_VALUE(a.dim() == 2 && w.dim() == (packed ? 1 : 2) && scale.dim() == 2, name,
                      packed ? ": a [m, k], packed [k*n*bits/8], scale [groups, n]" : ": a [m, k], b [k, n*bits/8], scale [groups, n] must be 2-D");
    TORCH_CHECK_TYPE(a.scalar_type() == at::kBFloat16 && scale.scalar_type() == at::kBFloat16 && w.scalar_type() == at::kByte, name,
                     ": a and scale must be bfloat16, the weights uint8");
    TORCH_CHECK_VALUE(bits == 8 || bits == 4, name, ": weight_bits must be 8 or 4");
    Shape s;
    s.m = a.size(0);
    s.k = a.size(1);
    s.n = packed ? scale.size(1) : w.size(1) * (8 / bits);
    TORCH_CHECK_VALUE(group >= 0, name, ": group_size must not be negative");
    const int64_t groups = group ? s.k / group : 1;
    const bool agree = scale.size(0) == groups && (packed ? w.numel() == s.k * s.n * bits / 8 : w.size(0) == s.k && scale.size(1) == s.n);
    TORCH_CHECK_VALUE(agree, name, ": shapes do not agree: a ", a.sizes(), ", weights ", w.sizes(), ", scale ", scale.sizes());
    if (bias.has_value())
        TORCH_CHECK_VALUE(bias->scalar_type() == at::kBFloat16 && bias->dim() == 1 && bias->size(0) == s.n, name, ": bias must be bfloat16 [n]");
    s.out_n = out_columns(s.n, activation);
    if (residual.has_value())
        TORCH_CHECK_VALUE(residual->scalar_type() == at::kBFloat16 && residual->dim() == 2 && residual->size(0) == s.m && residual->size(1) == s.out_n,
                          "bfaintb_gemm: residual must be bfloat16 [m, n]");
    return s;
}

template <bool PACKED>
Tensor gemm_on_gpu(const Tensor& a_in, const Tensor& w_in, const Tensor& scale_in, int64_t bits, int64_t group, const OptTensor& bias_in,
                   const OptTensor& residual_in, int64_t activation)
{
    const Shape s = check(a_in, w_in, scale_in, bits, group, bias_in, residual_in, activation, PACKED);
    const bool direct = a_in.stride(1) == 1 && a_in.stride(0) % 8 == 0 && reinterpret_cast<uintptr_t>(a_in.const_data_ptr()) % 16 == 0;
    const Tensor a = direct ? a_in : a_in.contiguous();
    const c10::MaybeOwned<Tensor> w = w_in.expect_contiguous(), scale = scale_in.expect_contiguous();
    const Tensor bias = bias_in.has_value() ? bias_in->contiguous() : Tensor();
    const Tensor residual = residual_in.has_value() ? residual_in->contiguous() : Tensor();
    const c10::DeviceGuard guard(a.device());
    Tensor c = at::empty({s.m, s.out_n}, a.options());
    if (s.m == 0 || s.n == 0) return c;
    const hipStream_t stream = c10::hip::getCurrentHIPStream(a.device().index()).stream();
    const uint32_t m = (uint32_t)s.m, n = (uint32_t)s.n, k = (uint32_t)s.k;
    const size_t need = PACKED ? bfaintb_gemm_prepacked_workspace_bytes(m, n, k, (int)bits, (uint32_t)group)
                               : bfaintb_gemm_workspace_bytes(m, n, k, (int)bits, (uint32_t)group);
    Tensor ws;
    if (need != 0) ws = workspaces().get((int64_t)need, a, stream);
    bfaintb_epilogue ep{};
    ep.bias = bias.defined() ? bias.const_data_ptr() : nullptr;
    ep.residual = residual.defined() ? residual.const_data_ptr() : nullptr;
    ep.ldr = (uint32_t)s.out_n;
    ep.activation = (uint32_t)activation;
    void* const wsp = need != 0 ? ws.data_ptr() : nullptr;
    const size_t ws_bytes = need != 0 ? (size_t)ws.numel() : 0;
    const uint32_t lda = (uint32_t)a.stride(0);
    const int rc = PACKED ? bfaintb_gemm_prepacked_fused(c.data_ptr(), a.const_data_ptr(), w->const_data_ptr(), scale->const_data_ptr(), &ep, m, n, k, lda,
                                                         (uint32_t)s.out_n, (int)bits, (uint32_t)group, wsp, ws_bytes, stream)
                          : bfaintb_gemm_fused(c.data_ptr(), a.const_data_ptr(), w->const_data_ptr(), scale->const_data_ptr(), &ep, m, n, k, lda, n,
                                               (uint32_t)s.out_n, (int)bits, (uint32_t)group, wsp, ws_bytes, stream);
    if (rc != 0) raise_library_error(rc, PACKED ? "bfaintb_gemm_prepacked" : "bfaintb_gemm");
    return c;
}

template <bool PACKED>
Tensor gemm_elsewhere(const Tensor& a, const Tensor& w, const Tensor& scale, int64_t bits, int64_t group, const OptTensor& bias, const OptTensor& residual,
                      int64_t activation)
{
    check(a, w, scale, bits, group, bias, residual, activation, PACKED);
    TORCH_CHECK(false, PACKED ? "bfaintb_gemm_prepacked" : "bfaintb_gemm", " runs on the GPU only (no CPU implementation)");
}

using OpSignature = Tensor(const Tensor&, const Tensor&, const Tensor&, int64_t, int64_t, const OptTensor&, const OptTensor&, int64_t);

template <bool PACKED>
const c10::TypedOperatorHandle<OpSignature>& op_handle()
{
    static const auto op = c10::Dispatcher::singleton()
                               .findSchemaOrThrow(PACKED ? "awesome_fusion::bfaintb_gemm_prepacked" : "awesome_fusion::bfaintb_gemm", "")
                               .typed<OpSignature>();
    return op;
}

// There is no backward formula: outputs that depend on something differentiable say so when asked for a gradient.
template <bool PACKED>
struct NoBackward : torch::autograd::Function<NoBackward<PACKED>> {
    static Tensor forward(torch::autograd::AutogradContext*, const Tensor& a, const Tensor& w, const Tensor& scale, int64_t bits, int64_t group,
                          const OptTensor& bias, const OptTensor& residual, int64_t activation)
    {
        at::AutoDispatchBelowADInplaceOrView below;
        return op_handle<PACKED>().call(a, w, scale, bits, group, bias, residual, activation);
    }
    static torch::autograd::variable_list backward(torch::autograd::AutogradContext*, torch::autograd::variable_list)
    {
        TORCH_CHECK(false, "Trying to backward through awesome_fusion::bfaintb_gemm", PACKED ? "_prepacked" : "", ", which has no autograd formula");
    }
};

template <bool PACKED>
Tensor gemm_autograd(const Tensor& a, const Tensor& w, const Tensor& scale, int64_t bits, int64_t group, const OptTensor& bias, const OptTensor& residual,
                     int64_t activation)
{
    const auto wants = [](const OptTensor& t) { return t.has_value() && t->requires_grad(); };
    if (c10::GradMode::is_enabled() && (a.requires_grad() || w.requires_grad() || scale.requires_grad() || wants(bias) || wants(residual)))
        return NoBackward<PACKED>::apply(a, w, scale, bits, group, bias, residual, activation);
    at::AutoDispatchBelowADInplaceOrView below;
    return op_handle<PACKED>().call(a, w, scale, bits, group, bias, residual, activation);
}

TORCH_LIBRARY(awesome_fusion, lib)
{
    lib.def("bfaintb_gemm(Tensor a, Tensor b, Tensor scale, int weight_bits, int group_size, Tensor? bias=None, Tensor? residual=None, int activation=0) -> Tensor",
            {at::Tag::pt2_compliant_tag});
    lib.def("bfaintb_gemm_prepacked(Tensor a, Tensor packed, Tensor scale, int weight_bits, int group_size, Tensor? bias=None, Tensor? residual=None, int activation=0) -> Tensor",
            {at::Tag::pt2_compliant_tag});
}
TORCH_LIBRARY_IMPL(awesome_fusion, CUDA, lib)
{
    lib.impl("bfaintb_gemm", gemm_on_gpu<false>);
    lib.impl("bfaintb_gemm_prepacked", gemm_on_gpu<true>);
}
TORCH_LIBRARY_IMPL(awesome_fusion, CPU, lib)
{
    lib.impl("bfaintb_gemm", gemm_elsewhere<false>);
    lib.impl("bfaintb_gemm_prepacked", gemm_elsewhere<true>);
}
TORCH_LIBRARY_IMPL(awesome_fusion, Autograd, lib)
{
    lib.impl("bfaintb_gemm", gemm_autograd<false>);
    lib.impl("bfaintb_gemm_prepacked", gemm_autograd<true>);
}

// ---- the module's functions, METH_FASTCALL

struct Names {
    PyObject *buffers, *parameters, *qweight, *scales, *bias, *weight_bits, *group_size, *prepacked, *in_features, *out_features;
} g_names;

// A tensor or Parameter itself: nothing that could override __torch_function__.
bool plain_tensor(PyObject* o) { return o != nullptr && THPVariable_CheckTypeExact(Py_TYPE(o)); }

// linear_forward(layer.__dict__, x, residual) -> y, or NotImplemented where the layer or an argument is not what this
// shortcut knows (overridden attributes, tensor subclasses, tracing proxies): the caller then takes the long way.
PyObject* linear_forward(PyObject*, PyObject* const* args, Py_ssize_t nargs)
{
    HANDLE_TH_ERRORS
    // (torch.jit.trace writes sizes read here down as constants: the long way's stay those of the input)
    if (nargs != 3 || !PyDict_Check(args[0]) || !plain_tensor(args[1]) || at::impl::torch_function_mode_enabled() || torch::jit::tracer::isTracing())
        Py_RETURN_NOTIMPLEMENTED;
    PyObject* const d = args[0];
    PyObject* const buffers = PyDict_GetItem(d, g_names.buffers);
    PyObject* const parameters = PyDict_GetItem(d, g_names.parameters);
    if (buffers == nullptr || parameters == nullptr || !PyDict_Check(buffers) || !PyDict_Check(parameters)) Py_RETURN_NOTIMPLEMENTED;
    PyObject* const qweight = PyDict_GetItem(buffers, g_names.qweight);
    PyObject* const scales = PyDict_GetItem(buffers, g_names.scales);
    PyObject* bias = PyDict_GetItem(parameters, g_names.bias);
    if (bias == nullptr) bias = PyDict_GetItem(d, g_names.bias);
    PyObject* const prepacked = PyDict_GetItem(d, g_names.prepacked);
    PyObject* const numbers[4] = {PyDict_GetItem(d, g_names.weight_bits), PyDict_GetItem(d, g_names.group_size), PyDict_GetItem(d, g_names.in_features),
                                  PyDict_GetItem(d, g_names.out_features)};
    if (!plain_tensor(qweight) || !plain_tensor(scales) || bias == nullptr || (bias != Py_None && !plain_tensor(bias)) ||
        (args[2] != Py_None && !plain_tensor(args[2])) || (prepacked != Py_True && prepacked != Py_False))
        Py_RETURN_NOTIMPLEMENTED;
    for (PyObject* v : numbers)
        if (v == nullptr || !PyLong_CheckExact(v)) Py_RETURN_NOTIMPLEMENTED;
    const int64_t bits = PyLong_AsLongLong(numbers[0]), group = PyLong_AsLongLong(numbers[1]);
    const int64_t in = PyLong_AsLongLong(numbers[2]), out = PyLong_AsLongLong(numbers[3]);
    // (references of their own: the layer may change while the interpreter's lock is released)
    const Tensor x = THPVariable_Unpack(args[1]), w = THPVariable_Unpack(qweight), s = THPVariable_Unpack(scales);
    OptTensor b, r;
    if (bias != Py_None) b = THPVariable_Unpack(bias);
    if (args[2] != Py_None) r = THPVariable_Unpack(args[2]);
    const bool packed = prepacked == Py_True;
    Tensor y;
    {
        pybind11::gil_scoped_release release;
        const bool as_it_is = x.dim() == 2 && x.size(1) == in;
        Tensor x2 = as_it_is ? x : x.reshape({-1, in});
        if (x2.scalar_type() != at::kBFloat16) x2 = x2.to(at::kBFloat16);
        if (r.has_value()) {
            if (r->dim() != 2 || r->size(1) != out) r = r->reshape({-1, out});
            if (r->scalar_type() != at::kBFloat16) r = r->to(at::kBFloat16);
        }
        y = (packed ? op_handle<true>() : op_handle<false>()).call(x2, w, s, bits, group, b, r, 0);
        if (!as_it_is) {  // (also of two dimensions but another width: refused here, by the number of elements)
            auto shape = x.sizes().vec();
            if (shape.empty()) shape.push_back(out);
            shape.back() = out;
            y = y.reshape(shape);
        }
    }
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

// The device pointer of an argument.  WRITTEN: what the call writes to — a tensor that shares its memory with a lazy copy
// gets memory of its own first.
template <bool WRITTEN>
bool pointer_of(PyObject* o, const void** out)
{
    if (o == Py_None) {
        *out = nullptr;
        return true;
    }
    if (PyLong_Check(o)) {
        *out = PyLong_AsVoidPtr(o);
        return !PyErr_Occurred();
    }
    if (THPVariable_Check(o)) {
        const Tensor& t = THPVariable_Unpack(o);
        *out = WRITTEN ? t.mutable_data_ptr() : t.const_data_ptr();
        return true;
    }
    PyObject* const address = PyObject_CallMethod(o, "data_ptr", nullptr);  // (whatever else carries a device pointer)
    if (address == nullptr) return false;
    *out = PyLong_AsVoidPtr(address);
    Py_DECREF(address);
    return !PyErr_Occurred();
}

// gemm_call(packed, c, a, b, scale, bias, residual, ldr, activation, m, n, k, lda, ldb, ldc, weight_bits, group_size, workspace,
//           workspace_nbytes, stream, which, force_split_k) -> return code.  workspace_nbytes None: all of the workspace (0 for a
//           bare address); stream None: torch's current one on the current device.
PyObject* gemm_call(PyObject*, PyObject* const* args, Py_ssize_t nargs)
{
    HANDLE_TH_ERRORS
    if (nargs != 22) {
        PyErr_SetString(PyExc_TypeError, "gemm_call takes 22 arguments");
        return nullptr;
    }
    const void *c, *a, *b, *scale, *bias, *residual, *workspace;
    if (!pointer_of<true>(args[1], &c) || !pointer_of<false>(args[2], &a) || !pointer_of<false>(args[3], &b) || !pointer_of<false>(args[4], &scale) ||
        !pointer_of<false>(args[5], &bias) || !pointer_of<false>(args[6], &residual) || !pointer_of<true>(args[17], &workspace))
        return nullptr;
    uint32_t v[22] = {};
    for (int i : {7, 8, 9, 10, 11, 12, 13, 14, 15, 16, 20, 21}) {
        v[i] = (uint32_t)PyLong_AsUnsignedLongMask(args[i]);
        if (v[i] == (uint32_t)-1 && PyErr_Occurred()) return nullptr;
    }
    size_t ws_bytes = 0;
    if (args[18] != Py_None) {
        ws_bytes = PyLong_AsSize_t(args[18]);
        if (ws_bytes == (size_t)-1 && PyErr_Occurred()) return nullptr;
    } else if (THPVariable_Check(args[17])) {
        ws_bytes = THPVariable_Unpack(args[17]).nbytes();
    } else if (args[17] != Py_None && !PyLong_Check(args[17])) {  // (whatever else carries a device pointer, as above)
        size_t factors[2];
        for (int i = 0; i < 2; ++i) {
            PyObject* const value = PyObject_CallMethod(args[17], i == 0 ? "numel" : "element_size", nullptr);
            if (value == nullptr) return nullptr;
            factors[i] = PyLong_AsSize_t(value);
            Py_DECREF(value);
            if (factors[i] == (size_t)-1 && PyErr_Occurred()) return nullptr;
        }
        ws_bytes = factors[0] * factors[1];
    }
    void* stream = nullptr;
    if (args[19] == Py_None) stream = c10::hip::getCurrentHIPStream().stream();
    else {
        stream = PyLong_AsVoidPtr(args[19]);
        if (PyErr_Occurred()) return nullptr;
    }
    const bool packed = PyObject_IsTrue(args[0]) == 1;
    const int bits = (int)v[15], which = (int)v[20];
    int rc;
    {
        pybind11::gil_scoped_release release;
        void* const cp = const_cast<void*>(c);
        void* const wsp = const_cast<void*>(workspace);
        if (residual != nullptr || v[8] != 0) {
            bfaintb_epilogue ep{};
            ep.bias = bias;
            ep.residual = residual;
            ep.ldr = v[7];
            ep.activation = v[8];
            rc = packed ? bfaintb_gemm_prepacked_fused(cp, a, b, scale, &ep, v[9], v[10], v[11], v[12], v[14], bits, v[16], wsp, ws_bytes, stream)
                        : bfaintb_gemm_fused(cp, a, b, scale, &ep, v[9], v[10], v[11], v[12], v[13], v[14], bits, v[16], wsp, ws_bytes, stream);
        } else if (packed) {
            rc = bfaintb_gemm_prepacked_ex(cp, a, b, scale, bias, v[9], v[10], v[11], v[12], v[14], bits, v[16], wsp, ws_bytes, stream, which);
        } else if (bias != nullptr) {
            rc = bfaintb_gemm_bias(cp, a, b, scale, bias, v[9], v[10], v[11], v[12], v[13], v[14], bits, v[16], wsp, ws_bytes, stream);
        } else {
            rc = bfaintb_gemm_ex(cp, a, b, scale, v[9], v[10], v[11], v[12], v[13], v[14], bits, v[16], wsp, ws_bytes, stream, which, v[21]);
        }
    }
    return PyLong_FromLong(rc);
    END_HANDLE_TH_ERRORS
}

PyObject* set_error_class(PyObject*, PyObject* cls)
{
    Py_INCREF(cls);
    Py_XDECREF(g_error_class);
    g_error_class = cls;
    Py_RETURN_NONE;
}

PyObject* release_workspaces(PyObject*, PyObject*)
{
    HANDLE_TH_ERRORS
    workspaces().clear();
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

PyMethodDef g_methods[] = {
    {"linear_forward", (PyCFunction)(void (*)(void))linear_forward, METH_FASTCALL, "QuantLinear's forward pass, or NotImplemented"},
    {"gemm_call", (PyCFunction)(void (*)(void))gemm_call, METH_FASTCALL, "one call of the C ABI: its return code"},
    {"set_error_class", set_error_class, METH_O, "the exception raised for the library's error codes: cls(code, what)"},
    {"release_workspaces", release_workspaces, METH_NOARGS, "gives the operators' split-K workspaces back (those of graphs that are still there excepted)"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_torch_binding", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__torch_binding(void)
{
    g_names = {PyUnicode_InternFromString("_buffers"),    PyUnicode_InternFromString("_parameters"), PyUnicode_InternFromString("qweight"),
               PyUnicode_InternFromString("scales"),      PyUnicode_InternFromString("bias"),        PyUnicode_InternFromString("weight_bits"),
               PyUnicode_InternFromString("group_size"),  PyUnicode_InternFromString("prepacked"),   PyUnicode_InternFromString("in_features"),
               PyUnicode_InternFromString("out_features")};
    return PyModule_Create(&g_module);
}
