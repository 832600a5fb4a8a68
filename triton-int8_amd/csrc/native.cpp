// The host side of a layer call (ops.linear_call) as one Python call: outputs, workspace and argument block, then the library's entry
// points.  It makes the same allocations and calls as the Python that it stands in for.  Calls with anything out of the ordinary
// (subclasses of Tensor, other dtypes, tensors that are not on a GPU) return None and take the Python way, which says what is wrong.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ops/empty.h>
#include <ATen/detail/CUDAHooksInterface.h>
#include <ATen/ops/narrow.h>
#include <ATen/TracerMode.h>
#include <c10/core/impl/DeviceGuardImplInterface.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>

#include "../../include/ti8.h"

namespace {

// The library is the one that the binding has loaded: its entry points come from there
decltype(&ti8_linear) linear = nullptr;
decltype(&ti8_linear_quantise) linear_quantise = nullptr;
decltype(&ti8_gemm_i8_nt_multi) gemm_multi = nullptr;
PyObject* parameter_class = nullptr;

// *out = the tensor behind `o` (undefined for None); false if it is not a plain tensor
bool plain(PyObject* o, at::Tensor* out) {
    if (o == Py_None) return true;
    if (Py_TYPE(o) != reinterpret_cast<PyTypeObject*>(THPVariableClass) && Py_TYPE(o) != reinterpret_cast<PyTypeObject*>(parameter_class)) return false;
    *out = THPVariable_Unpack(o);
    return true;
}

bool bf16_matrix(const at::Tensor& t) { return !t.defined() || (t.is_cuda() && t.scalar_type() == at::kBFloat16 && t.dim() == 2); }

// The tensor itself where the library can read its rows in place, else a dense copy (ops.rows16)
at::Tensor rows16(const at::Tensor& t) {
    if (!t.defined()) return t;
    const int64_t row = t.stride(0);
    if (t.stride(1) == 1 && row % 8 == 0 && row >= t.size(1) && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0) return t;
    return t.clone(at::MemoryFormat::Contiguous);
}

struct GilReleased {
    PyThreadState* const state = PyEval_SaveThread();
    ~GilReleased() { PyEval_RestoreThread(state); }
};

// Device memory that a call needs until its launches are queued, from the allocator that tensors come from at the time (a program may put its own in
// the place of torch's) but without making one
struct Workspace {
    c10::DataPtr plain;
    at::Tensor tensor;
    void* p;
    Workspace(int64_t bytes, const at::Device& dev, const at::TensorOptions& options) {
        if (c10::impl::getDeviceGuardImpl(c10::DeviceType::CUDA)->getDevice() == dev) {
            plain = at::detail::getCUDAHooks().getCUDADeviceAllocator()->allocate(bytes);
            p = plain.get();
        } else {
            tensor = at::empty({bytes}, options);
            p = tensor.data_ptr();
        }
    }
};

// Whether a tracer, a dispatch mode or a function transform looks at the operators of this thread
bool followed() {
    return at::tracer::impl::is_dispatch_enabled() || c10::impl::dispatch_mode_enabled() ||
           c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode);
}

PyObject* wrap(const at::Tensor& t) {
    if (t.defined()) return THPVariable_Wrap(t);
    Py_RETURN_NONE;
}

enum { PARTS, SCHEME, HADAMARD, TOKENS, K_, N_, GEMM_FLAGS, NEED, NEED_SAVED, APART, STREAM, SERVED, NUMBERS, TENSORS = 7 };

// linear_call(parts, scheme, hadamard, tokens, K, N, gemm_flags, workspace bytes, saved bytes, whether the GEMMs are a call of their
// own, stream, whether only Y is wanted, and of that the rows of tokens alone, X, W, dY, wq, ws, saved, bias) -> (Y, dX, dW, saved) or that Y,
// (name, status) of an entry point that failed, or None
PyObject* linear_call(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (nargs != NUMBERS + TENSORS) {
        PyErr_SetString(PyExc_TypeError, "linear_call takes 19 arguments");
        return nullptr;
    }
    at::Tensor X, W, dY, wq, ws, saved, bias;
    at::Tensor* const tensors[TENSORS] = {&X, &W, &dY, &wq, &ws, &saved, &bias};
    for (int i = 0; i < TENSORS; ++i)
        if (!plain(args[NUMBERS + i], tensors[i])) Py_RETURN_NONE;
    if (!bf16_matrix(X) || !bf16_matrix(W) || !bf16_matrix(dY) || (!X.defined() && !dY.defined())) Py_RETURN_NONE;
    int64_t v[NUMBERS];
    for (int i = 0; i < NUMBERS; ++i) {
        v[i] = PyLong_AsLongLong(args[i]);
        if (v[i] == -1 && PyErr_Occurred()) return nullptr;
    }
    at::Tensor Y, dX, dW;
    const char* name = "ti8_linear";
    int status;
    {
        const GilReleased released;      // the allocator and the library have locks of their own
        const int64_t tokens = v[TOKENS], K = v[K_], N = v[N_], T = (tokens + 127) / 128 * 128;
        const at::Device dev = X.defined() ? X.device() : dY.device();
        const auto bf16 = at::TensorOptions().dtype(at::kBFloat16).device(dev), bytes = at::TensorOptions().dtype(at::kByte).device(dev);
        X = rows16(X);
        W = rows16(W);
        dY = rows16(dY);
        if (v[PARTS] & TI8_PART_FORWARD) {
            Y = at::empty({T, N}, bf16);
            if (v[NEED_SAVED]) saved = at::empty({v[NEED_SAVED]}, bytes);
        }
        if (v[PARTS] & TI8_PART_BACKWARD) {
            dX = at::empty({T, K}, bf16);
            dW = at::empty({N, K}, bf16);
        }
        const Workspace workspace(v[NEED], dev, bytes);
        const auto ptr = [](const at::Tensor& t) -> void* { return t.defined() ? t.data_ptr() : nullptr; };
        const auto row = [](const at::Tensor& t) -> int64_t { return t.defined() ? t.stride(0) : 0; };
        ti8_linear_args a = {};
        a.X = ptr(X); a.ldx = row(X);
        a.W = ptr(W); a.ldw = row(W);
        a.dY = ptr(dY); a.lddy = row(dY);
        a.Y = ptr(Y); a.ldy = N;
        a.dX = ptr(dX); a.lddx = K;
        a.dW = ptr(dW); a.lddw = K;
        a.wq = static_cast<const int8_t*>(ptr(wq)); a.ws = static_cast<const float*>(ptr(ws));
        a.tokens = tokens; a.K = K; a.N = N;
        a.scheme = (int)v[SCHEME]; a.hadamard = (int)v[HADAMARD]; a.parts = (int)v[PARTS]; a.gemm_flags = (int)v[GEMM_FLAGS];
        a.workspace = workspace.p; a.workspace_bytes = v[NEED];      // (device allocations start on 512-byte boundaries)
        a.saved = ptr(saved); a.saved_bytes = v[NEED_SAVED];
        a.bias = ptr(bias);
        ti8_stream_t stream = reinterpret_cast<ti8_stream_t>(static_cast<uintptr_t>(v[STREAM]));
        if (v[APART]) {
            ti8_gemm_problem problems[3];
            int count = 0;
            name = "ti8_linear_quantise";
            status = linear_quantise(&a, problems, &count, stream);
            if (status == TI8_OK) {
                name = "ti8_gemm_i8_nt_multi";
                status = gemm_multi(problems, count, a.gemm_flags | TI8_GEMM_TOGETHER, stream);
            }
        } else {
            status = linear(&a, stream);
        }
    }
    if (status != TI8_OK) return Py_BuildValue("(si)", name, status);
    if (v[SERVED]) {
        // (in its own sizes, unless something follows what is made of Y operator by operator)
        if (followed()) Y = Y.narrow(0, 0, v[TOKENS]);
        else Y.unsafeGetTensorImpl()->set_sizes_contiguous({v[TOKENS], v[N_]});
        return wrap(Y);
    }
    return Py_BuildValue("(NNNN)", wrap(Y), wrap(dX), wrap(dW), wrap(saved));
    END_HANDLE_TH_ERRORS
}

// set_up(addresses of ti8_linear, ti8_linear_quantise, ti8_gemm_i8_nt_multi; torch.nn.Parameter)
PyObject* set_up(PyObject*, PyObject* args) {
    unsigned long long l, q, g;
    PyObject* parameter;
    if (!PyArg_ParseTuple(args, "KKKO", &l, &q, &g, &parameter)) return nullptr;
    linear = reinterpret_cast<decltype(linear)>(l);
    linear_quantise = reinterpret_cast<decltype(linear_quantise)>(q);
    gemm_multi = reinterpret_cast<decltype(gemm_multi)>(g);
    Py_INCREF(parameter);
    Py_XSETREF(parameter_class, parameter);
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"linear_call", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(linear_call)), METH_FASTCALL, nullptr},
    {"set_up", set_up, METH_VARARGS, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// built_for: what the code above was compiled against, for whoever loads it to compare (fields of torch's and Python's objects and of the
// library's argument blocks are read and written here without a call)
PyMODINIT_FUNC PyInit__native(void) {
    PyObject* const m = PyModule_Create(&module);
    PyObject* const built_for = Py_BuildValue("(s(ii)nn)", TI8_BUILT_FOR_TORCH, PY_MAJOR_VERSION, PY_MINOR_VERSION, (Py_ssize_t)sizeof(ti8_linear_args), (Py_ssize_t)sizeof(ti8_gemm_problem));
    if (m && (!built_for || PyModule_AddObject(m, "built_for", built_for) < 0)) {
        Py_XDECREF(built_for);
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
