// The eager host path of the small calls (one linear, one norm, one
// activation): a decode step is bound by what the host does per call, about
// 9 us from Python of which the kernel launch is 3.  Each function here takes
// the module's tensors, makes the checks, allocates the outputs and calls the
// C entry point in one step; whatever is not the plain case (another type,
// layout or device, a tensor subclass, an active mode or transform, graph
// capture, a workspace that must grow, an argument the entry point refuses
// before it launches anything) returns None and the caller takes its Python
// path, which handles it or raises.  An error after a launch raises here: the
// call is never made a second time.  Figures stand at the callers.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <utility>

#include "kbn_fp8.h"

namespace {

constexpr int64_t kGroup = 128;
constexpr float kQuantEps = 1e-10f;

// Nothing watches or replaces tensor operations on this thread.
bool plain_thread() {
    return !c10::impl::TorchDispatchModeTLS::any_modes_set() &&
           at::impl::PythonTorchFunctionTLS::stack_len() == 0 &&
           !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode);
}

// A torch.Tensor or Parameter itself (no subclass), strided, on a GPU.
const at::Tensor* plain_tensor(PyObject* o) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    return t.defined() && t.is_cuda() && t.layout() == at::kStrided ? &t : nullptr;
}

bool is(const at::Tensor& t, at::ScalarType type, int64_t dev, int64_t dim) {
    return t.scalar_type() == type && t.get_device() == dev && t.dim() == dim;
}

// The launch stream of device dev, which must be the current one and not be
// capturing a graph.
bool launch_stream(int64_t dev, hipStream_t& st) {
    if (c10::hip::current_device() != dev) return false;
    st = c10::hip::getCurrentHIPStream((c10::DeviceIndex)dev).stream();
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(st, &cs) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return cs == hipStreamCaptureStatusNone;
}

at::Tensor empty_codes(const at::Tensor& like, int64_t rows, int64_t cols) {
    return at::empty({rows, cols}, like.options().dtype(at::kFloat8_e4m3fn).requires_grad(false));
}
at::Tensor empty_scales(const at::Tensor& like, int64_t rows, int64_t groups) {   // column-major
    return at::empty_strided({rows, groups}, {1, rows}, like.options().dtype(at::kFloat).requires_grad(false));
}

// An eager workspace of at least `bytes` for (device, stream), from the dict
// the Python side keeps ({(device, stream): uint8 tensor}); undefined if it
// has none that large.  The caller holds the tensor over its launch: another
// thread may put a larger one in its place once the GIL is released.
at::Tensor kept_workspace(PyObject* bufs, int64_t dev, hipStream_t st, int64_t bytes) {
    PyObject* key = Py_BuildValue("(LL)", (long long)dev, (long long)(intptr_t)st);
    if (!key) {
        PyErr_Clear();
        return {};
    }
    PyObject* buf = PyDict_GetItem(bufs, key);   // borrowed; no exception set
    Py_DECREF(key);
    const at::Tensor* t = buf ? plain_tensor(buf) : nullptr;
    return t && t->numel() >= bytes ? *t : at::Tensor();
}

// No GIL while it lives; taken again on every way out, an exception included
// (guarded below calls into Python).
struct NoGil {
    PyThreadState* s = PyEval_SaveThread();
    ~NoGil() { PyEval_RestoreThread(s); }
};

// Failures of the torch calls (out of memory, say) surface from the Python path.
template <class F>
PyObject* guarded(F&& f) {
    try {
        return f();
    } catch (...) {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
}

// What a call that ended with `rc` != 0 gives.  1: an argument was refused and
// nothing was launched, so None, and the Python path refuses it too.  Anything
// else comes after a launch (the runtime's last error, which may be another
// call's): the launch may have run, and a fused add + norm run again would add
// twice, so the error is raised as the Python path raises it.
PyObject* failed(int rc, const char* what) {
    if (rc == 1) Py_RETURN_NONE;
    if (PyObject* lib = PyImport_ImportModule("kb_nano_amd._lib")) {
        PyObject* r = PyObject_CallMethod(lib, "check", "is", rc, what);   // raises KbnError
        Py_DECREF(lib);
        Py_XDECREF(r);
    }
    if (!PyErr_Occurred()) PyErr_Format(PyExc_RuntimeError, "%s failed (code %d)", what, rc);
    return nullptr;
}

// failed(code, name): the rule above, for tests
PyObject* failed_call(PyObject*, PyObject* const* args, Py_ssize_t n) {
    const char* what = n == 2 ? PyUnicode_AsUTF8(args[1]) : nullptr;
    const long rc = what ? PyLong_AsLong(args[0]) : 0;
    if (!what || PyErr_Occurred()) return PyErr_Format(PyExc_TypeError, "failed(code, name)");
    return failed((int)rc, what);
}

// (codes, scales), made before the launch so that nothing but the launch can
// fail after it; empty with the Python error set if it cannot be made.
struct Ref {
    PyObject* p;
    ~Ref() { Py_XDECREF(p); }
    PyObject* take() { return std::exchange(p, nullptr); }
};
PyObject* pair(const at::Tensor& q, const at::Tensor& s) {
    Ref a{THPVariable_Wrap(q)}, b{THPVariable_Wrap(s)};
    return a.p && b.p ? PyTuple_Pack(2, a.p, b.p) : nullptr;
}

// norm(input, weight, eps, residual | None) -> (codes, scales) | None
PyObject* norm(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 4) Py_RETURN_NONE;
    return guarded([&]() -> PyObject* {
        const bool add = args[3] != Py_None;
        const at::Tensor *x = plain_tensor(args[0]), *w = plain_tensor(args[1]), *r = add ? plain_tensor(args[3]) : nullptr;
        if (!x || !w || (add && !r) || !PyFloat_CheckExact(args[2]) || !plain_thread()) Py_RETURN_NONE;
        const int64_t dev = x->get_device();
        hipStream_t st;
        if (x->dim() < 1 || x->numel() == 0 || !is(*x, at::kBFloat16, dev, x->dim()) || !is(*w, at::kBFloat16, dev, 1) ||
            !x->is_contiguous() || !w->is_contiguous() || !launch_stream(dev, st))
            Py_RETURN_NONE;
        const int64_t H = x->size(-1), T = x->numel() / H;
        if (w->size(0) != H || (add && (!is(*r, at::kBFloat16, dev, x->dim()) || !r->is_contiguous() ||
                                        r->sizes() != x->sizes())))
            Py_RETURN_NONE;
        const at::Tensor q = empty_codes(*x, T, H), s = empty_scales(*x, T, (H + kGroup - 1) / kGroup);
        Ref out{pair(q, s)};
        if (!out.p) return nullptr;
        int rc;
        {
            NoGil no_gil;
            rc = kbn_rmsnorm_fp8_quant(x->data_ptr(), T, H, H, w->data_ptr(), add ? r->data_ptr() : nullptr, H, q.data_ptr(),
                                       H, (float*)s.data_ptr(), s.stride(0), s.stride(1), (float)PyFloat_AS_DOUBLE(args[2]),
                                       (void*)st);
        }
        if (rc) return failed(rc, add ? "fused_add_rmsnorm_fp8_quant" : "rmsnorm_fp8_quant");
        return out.take();
    });
}

// silu(input, ue8m0, eps) -> (codes, scales) | None
PyObject* silu(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 3) Py_RETURN_NONE;
    return guarded([&]() -> PyObject* {
        const at::Tensor* x = plain_tensor(args[0]);
        if (!x || !PyFloat_CheckExact(args[2]) || !plain_thread()) Py_RETURN_NONE;
        const int ue8m0 = PyObject_IsTrue(args[1]);   // any object, as in Python: its truth value may raise
        if (ue8m0 < 0) return nullptr;
        const int64_t dev = x->get_device();
        hipStream_t st;
        if (!is(*x, at::kBFloat16, dev, 2) || x->numel() == 0 || x->stride(1) != 1 || !launch_stream(dev, st))
            Py_RETURN_NONE;
        const int64_t M = x->size(0), Nh = x->size(1) / 2;
        if (M % kGroup || Nh % kGroup || x->size(1) % 2) Py_RETURN_NONE;
        const at::Tensor q = empty_codes(*x, M, Nh), s = empty_scales(*x, M, Nh / kGroup);
        Ref out{pair(q, s)};
        if (!out.p) return nullptr;
        int rc;
        {
            NoGil no_gil;
            rc = kbn_silu_mul_quant_fp8(x->data_ptr(), M, Nh, x->stride(0), q.data_ptr(), Nh, (float*)s.data_ptr(), s.stride(0),
                                        s.stride(1), (float)PyFloat_AS_DOUBLE(args[2]), ue8m0, (void*)st);
        }
        if (rc) return failed(rc, "silu_mul_quant_fp8");
        return out.take();
    });
}

// Whether a shape's bf16-input GEMM is preferred, and its workspace: the
// thread's latest answers, as each asks for a plan.
struct Bf16aPlan {
    int64_t M = 0, N = 0, K = 0, dev = -1;
    bool preferred = false;
    int64_t ws = 0;
};
const Bf16aPlan& bf16a_plan(int64_t dev, int64_t M, int64_t N, int64_t K) {
    thread_local Bf16aPlan kept[64];
    Bf16aPlan& p = kept[(uint64_t)(M * 31 + N * 7 + K / 128 + dev) % 64];
    if (p.M != M || p.N != N || p.K != K || p.dev != dev) {
        p.preferred = kbn_fp8_gemm_bf16a_preferred(M, N, K) != 0;
        p.ws = p.preferred ? kbn_fp8_gemm_bf16a_workspace_bytes(M, N, K) : 0;
        p.M = M; p.N = N; p.K = K; p.dev = dev;
    }
    return p;
}

// linear(x, weight, weight_scale, a_buf | None, s_buf | None, o_buf | None,
//        prefill buffers | None, ue8m0, workspaces) -> output [M, N] | None
PyObject* linear(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 9) Py_RETURN_NONE;
    return guarded([&]() -> PyObject* {
        const at::Tensor *x = plain_tensor(args[0]), *w = plain_tensor(args[1]), *ws = plain_tensor(args[2]);
        if (!x || !w || !ws || !PyDict_CheckExact(args[8]) || !plain_thread()) Py_RETURN_NONE;
        const int64_t dev = x->get_device();
        hipStream_t st;
        if (!is(*x, at::kBFloat16, dev, 2) || !is(*w, at::kFloat8_e4m3fn, dev, 2) || !is(*ws, at::kFloat, dev, 2) ||
            x->numel() == 0 || w->numel() == 0 || !launch_stream(dev, st))
            Py_RETURN_NONE;
        const int64_t M = x->size(0), K = x->size(1), N = w->size(0);
        if (w->size(1) != K || K % kGroup || ws->size(0) * kGroup < N || ws->size(1) * kGroup < K || x->stride(1) != 1 ||
            w->stride(1) != 1 || ws->stride(1) != 1)
            Py_RETURN_NONE;
        // the installed buffers that hold M rows: decode, else prefill
        const bool ue8m0 = PyObject_IsTrue(args[7]) == 1;
        const Bf16aPlan* direct = M <= 64 && ue8m0 ? &bf16a_plan(dev, M, N, K) : nullptr;
        if (direct && !direct->preferred) direct = nullptr;
        PyObject* const pf = args[6];
        PyObject *qo = args[3], *so = args[4], *oo = args[5];
        auto rows = [](PyObject* o) { const at::Tensor* t = plain_tensor(o); return t && t->dim() == 2 ? t->size(0) : -1; };
        PyObject* held[3] = {nullptr, nullptr, nullptr};   // attributes of pf
        struct Release {
            PyObject** h;
            ~Release() { for (int i = 0; i < 3; ++i) Py_XDECREF(h[i]); }
        } release{held};
        if (rows(direct ? oo : qo) < M) {
            if (pf == Py_None) Py_RETURN_NONE;
            const char* names[3] = {"a", "s", "o"};
            for (int i = 0; i < 3; ++i)
                if (!(held[i] = PyObject_GetAttrString(pf, names[i]))) {
                    PyErr_Clear();
                    Py_RETURN_NONE;
                }
            qo = held[0]; so = held[1]; oo = held[2];
        }
        const at::Tensor* o = plain_tensor(oo);
        if (!o || !is(*o, at::kBFloat16, dev, 2) || o->size(0) < M || o->size(1) != N || o->stride(1) != 1) Py_RETURN_NONE;
        int rc;
        if (direct) {
            const int64_t bytes = direct->ws;
            const at::Tensor buf = bytes ? kept_workspace(args[8], dev, st, bytes) : at::Tensor();
            if (bytes && !buf.defined()) Py_RETURN_NONE;
            void* const wsp = bytes ? buf.data_ptr() : nullptr;
            {
                NoGil no_gil;
                rc = kbn_fp8_gemm_bf16a(x->data_ptr(), x->stride(0), kQuantEps, w->data_ptr(), w->stride(0),
                                        (const float*)ws->data_ptr(), ws->stride(0), o->data_ptr(), o->stride(0), M, N, K, wsp,
                                        bytes, (void*)st);
            }
        } else {
            const at::Tensor *q = plain_tensor(qo), *s = plain_tensor(so);
            if (!q || !s || !is(*q, at::kFloat8_e4m3fn, dev, 2) || !is(*s, at::kFloat, dev, 2) || q->size(0) < M ||
                q->size(1) != K || q->stride(1) != 1 || s->size(0) < M || s->size(1) != K / kGroup)
                Py_RETURN_NONE;
            const int64_t bytes = kbn_fp8_gemm_nt_workspace_bytes(M, N, K, ue8m0);
            const at::Tensor buf = bytes ? kept_workspace(args[8], dev, st, bytes) : at::Tensor();
            if (bytes && !buf.defined()) Py_RETURN_NONE;
            void* const wsp = bytes ? buf.data_ptr() : nullptr;
            {
                NoGil no_gil;
                rc = kbn_fp8_linear_forward(x->data_ptr(), M, K, x->stride(0), q->data_ptr(), q->stride(0),
                                            (float*)s->data_ptr(), s->stride(0), s->stride(1), kQuantEps, 1, w->data_ptr(),
                                            w->stride(0), (const float*)ws->data_ptr(), ws->stride(0), o->data_ptr(),
                                            o->stride(0), N, ue8m0, wsp, bytes, (void*)st);
            }
        }
        if (rc) return failed(rc, direct ? "fp8_gemm_bf16a" : "fp8_linear_forward");
        if (o->size(0) == M) {
            Py_INCREF(oo);
            return oo;
        }
        return THPVariable_Wrap(o->narrow(0, 0, M));
    });
}

PyMethodDef kMethods[] = {
    {"norm", (PyCFunction)(void (*)())norm, METH_FASTCALL, "RMSNorm (+ residual add) + 1x128 quant"},
    {"silu", (PyCFunction)(void (*)())silu, METH_FASTCALL, "SiLU*Mul + 1x128 quant"},
    {"linear", (PyCFunction)(void (*)())linear, METH_FASTCALL, "bf16 activations through an FP8 weight"},
    {"failed", (PyCFunction)(void (*)())failed_call, METH_FASTCALL, "what a call gives for an error code"},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) { return PyModule_Create(&kModule); }
