// Native front end of the Python binding: flash_attn_amd._native.
//
// flash_forward / flash_forward_splitkv of binding.py hand their arguments to the two functions below, which fill
// flash_params, allocate the results and call the C ABI (the launch path of the reference's main(), src/main.cu:109-192).
//
// What bounds a small call is this code: filling the struct field by field through ctypes, five data_ptr() calls, two
// torch.empty() and torch.cuda.current_stream() took 13-15 us of host time per flash_forward and 18-19 us per
// flash_forward_splitkv, where the kernel of a small problem (B1 H2 N128 d64) runs for 4.6 us.
//
// Anything out of the ordinary -- an argument of another type, shapes or dtypes that do not fit, a workspace that is too
// small, a program that wants to see its allocations -- returns NotImplemented with nothing allocated or launched; binding.py then takes its own path, which raises the
// errors (and serves the debug outputs).
#include <torch/csrc/autograd/python_variable.h>
#include <torch/version.h>

#include <ATen/Context.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime.h>

#include <cmath>

#include "flash_attn_mi355.h"
#include "split_counters.h"

namespace {

typedef int (*launch_fn)(const flash_params*, void*);
typedef int (*resolve_fn)(const flash_params*);
launch_fn g_forward = nullptr, g_splitkv = nullptr;
resolve_fn g_resolve = nullptr;
PyObject* g_error = nullptr;  // binding.FlashError(code, where)

PyObject* not_implemented() { Py_RETURN_NOTIMPLEMENTED; }

// an ordinary tensor (no subclass with behaviour of its own), or nullptr
const at::Tensor* tensor_of(PyObject* o) { return THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr; }

bool fp16_on_gpu(const at::Tensor& t) { return t.scalar_type() == at::kHalf && t.is_cuda() && t.dim() == 4 && t.is_contiguous(); }

enum Parsed { kOk, kPython, kRaised };

// an exact int that fits the C int; anything else is left to binding.py
bool small_int(PyObject* o, int* out)
{
    if (!PyLong_CheckExact(o)) return false;
    int over = 0;
    const long v = PyLong_AsLongAndOverflow(o, &over);
    if (over != 0 || v < INT32_MIN || v > INT32_MAX) return false;
    *out = (int)v;
    return true;
}

bool real(PyObject* o, float* out)
{
    if (PyFloat_CheckExact(o)) {
        *out = (float)PyFloat_AS_DOUBLE(o);
        return true;
    }
    if (!PyLong_CheckExact(o)) return false;
    const double v = PyLong_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) {
        PyErr_Clear();
        return false;
    }
    *out = (float)v;
    return true;
}

bool optional_tensor(PyObject* o, const at::Tensor** t)
{
    *t = nullptr;
    return o == Py_None || (*t = tensor_of(o)) != nullptr;
}

// What the table of split_counters.h asks for.  A region is 16 KiB of the stream's own pool, kept until the process ends, at
// most 1 MiB per device.  (All of this runs with the interpreter lock held.)
struct TorchRuntime {
    int current_device() const
    {
        int d = -1;
        return hipGetDevice(&d) == hipSuccess ? d : -1;
    }
    bool capturing(void* stream) const
    {
        hipStreamCaptureStatus c;
        return hipStreamIsCapturing(static_cast<hipStream_t>(stream), &c) != hipSuccess || c != hipStreamCaptureStatusNone;
    }
    uint32_t* allocate(size_t words, void* stream) const
    {
        try {
            return static_cast<uint32_t*>(
                c10::hip::HIPCachingAllocator::raw_alloc_with_stream(words * sizeof(uint32_t), static_cast<hipStream_t>(stream)));
        } catch (const c10::Error&) {
            return nullptr;
        }
    }
    void release(uint32_t* p) const { c10::hip::HIPCachingAllocator::raw_delete(p); }
    bool clear(uint32_t* p, size_t words, void* stream) const
    {
        return hipMemsetAsync(p, 0, words * sizeof(uint32_t), static_cast<hipStream_t>(stream)) == hipSuccess;
    }
};
uint32_t* counters_of(at::Device device, void* stream, bool pooled)
{
    static auto* table = new fa::CounterTable<TorchRuntime>;  // (never freed: outlives the runtime's own end)
    TorchRuntime rt;
    return table->of(rt, device.index(), stream, pooled);
}

struct Call {
    flash_params p{};
    const at::Tensor* q = nullptr;
    const at::Tensor *out = nullptr, *lse = nullptr;
    void* stream = nullptr;
    bool pooled_stream = false;  // one of torch's own
};

// Results and workspace come from the allocator directly: through the dispatcher each takes 0.2 us more (B1 H2 N128 d64, whose
// call is bound by its host time: 5.07 against 5.47 us).  Who would notice gets torch.empty() instead: dispatch modes (fake tensors, tracers, memory accounting), and the
// deterministic mode that fills new memory.
bool allocates_plainly()
{
    return !c10::impl::TorchDispatchModeTLS::any_modes_set() &&
           !(at::globalContext().deterministicAlgorithms() && at::globalContext().deterministicFillUninitializedMemory());
}

// Arguments that both entry points share: q, k, v and the array (softmax_scale, causal, window, alibi_slopes, dropout_p,
// seed, offset, stream, out, lse).
Parsed parse(PyObject* const* qkv, PyObject* const* a, Call* c)
{
    if (!allocates_plainly()) return kPython;
    const at::Tensor *q = tensor_of(qkv[0]), *k = tensor_of(qkv[1]), *v = tensor_of(qkv[2]), *slopes;
    if (!q || !k || !v || !fp16_on_gpu(*q) || !fp16_on_gpu(*k) || !fp16_on_gpu(*v)) return kPython;
    const auto qs = q->sizes(), ks = k->sizes();
    if (ks[0] != qs[0] || ks[1] < 1 || qs[1] % ks[1] != 0 || ks[3] != qs[3] || v->sizes() != ks) return kPython;
    for (int i = 0; i < 4; ++i)
        if (qs[i] > INT32_MAX || ks[i] > INT32_MAX) return kPython;
    flash_params& p = c->p;
    p.B = (int)qs[0], p.H = (int)qs[1], p.Nq = (int)qs[2], p.d = (int)qs[3], p.H_kv = (int)ks[1], p.Nk = (int)ks[2];
    if (a[0] == Py_None) p.softmax_scale = (float)std::pow((double)p.d, -0.5);
    else if (!real(a[0], &p.softmax_scale)) return kPython;
    const int causal = PyObject_IsTrue(a[1]);
    if (causal < 0) return kRaised;
    p.is_causal = causal;
    if (!PyTuple_CheckExact(a[2]) || PyTuple_GET_SIZE(a[2]) != 2 || !small_int(PyTuple_GET_ITEM(a[2], 0), &p.window_left) ||
        !small_int(PyTuple_GET_ITEM(a[2], 1), &p.window_right))
        return kPython;
    if (!optional_tensor(a[3], &slopes)) return kPython;
    if (!real(a[4], &p.dropout_p) || !PyLong_CheckExact(a[5]) || !PyLong_CheckExact(a[6])) return kPython;
    p.seed = PyLong_AsUnsignedLongLongMask(a[5]);
    p.offset = PyLong_AsUnsignedLongLongMask(a[6]);
    if (!optional_tensor(a[8], &c->out) || !optional_tensor(a[9], &c->lse)) return kPython;
    if (a[7] == Py_None) {
        const auto current = c10::hip::getCurrentHIPStream();
        c->stream = current.stream();
        c->pooled_stream = (current.id() & 1) != 0;  // (the id of a stream from outside is its handle, an aligned pointer)
    } else {
        PyObject* h = PyObject_GetAttrString(a[7], "cuda_stream");
        if (!h) return kRaised;
        c->stream = PyLong_AsVoidPtr(h);
        Py_DECREF(h);
        if (PyErr_Occurred()) return kRaised;
        if (PyObject* id = PyObject_GetAttrString(a[7], "stream_id")) {
            c->pooled_stream = PyLong_Check(id) && (PyLong_AsUnsignedLongLongMask(id) & 1) != 0;
            Py_DECREF(id);
        } else {
            PyErr_Clear();
        }
    }
    p.Q = q->data_ptr(), p.K = k->data_ptr(), p.V = v->data_ptr();
    p.alibi_slopes = slopes ? static_cast<const float*>(slopes->data_ptr()) : nullptr;
    c->q = q;
    return kOk;
}

at::Tensor empty_like_q(const Call& c, at::IntArrayRef size, at::ScalarType type)
{
    return at::detail::empty_cuda(size, type, c.q->device(), std::nullopt);
}

PyObject* raise(int code, const char* where)
{
    PyObject* e = PyObject_CallFunction(g_error, "is", code, where);
    if (e) {
        PyErr_SetObject(g_error, e);
        Py_DECREF(e);
    }
    return nullptr;
}

// allocates what the caller has not brought, launches, returns (O, LSE)
PyObject* launch(launch_fn fn, const char* where, Call* c)
{
    flash_params& p = c->p;
    const at::Tensor o = c->out ? *c->out : empty_like_q(*c, c->q->sizes(), at::kHalf);
    const at::Tensor l = c->lse ? *c->lse : empty_like_q(*c, {p.B, p.H, p.Nq}, at::kFloat);
    p.O = o.data_ptr();
    p.LSE = static_cast<float*>(l.data_ptr());
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = fn(&p, c->stream);
    Py_END_ALLOW_THREADS
    if (rc != FLASH_OK) return raise(rc, where);
    PyObject* res = PyTuple_New(2);
    if (!res) return nullptr;
    PyTuple_SET_ITEM(res, 0, THPVariable_Wrap(o));
    PyTuple_SET_ITEM(res, 1, THPVariable_Wrap(l));
    return res;
}

// A C++ exception (an allocation that does not fit) becomes the Python exception that torch.empty would have raised.
template <typename F>
PyObject* guarded(F f)
{
    HANDLE_TH_ERRORS
    return f();
    END_HANDLE_TH_ERRORS
}

// forward(q, k, v, softmax_scale, causal, window, alibi_slopes, dropout_p, seed, offset, stream, out, lse)
PyObject* forward(PyObject*, PyObject* const* args, Py_ssize_t n)
{
    return guarded([&]() -> PyObject* {
        if (n != 13 || !g_forward) return not_implemented();
        Call c;
        const Parsed r = parse(args, args + 3, &c);
        if (r != kOk) return r == kPython ? not_implemented() : nullptr;
        c.p.num_splits = 1;
        return launch(g_forward, "flash_forward", &c);
    });
}

// splitkv(q, k, v, num_splits, workspace, softmax_scale, causal, window, alibi_slopes, dropout_p, seed, offset, stream,
// out, lse)
PyObject* splitkv(PyObject*, PyObject* const* args, Py_ssize_t n)
{
    return guarded([&]() -> PyObject* {
        if (n != 15 || !g_splitkv) return not_implemented();
        Call c;
        int splits;
        if (!small_int(args[3], &splits)) return not_implemented();
        const Parsed r = parse(args, args + 5, &c);
        if (r != kOk) return r == kPython ? not_implemented() : nullptr;
        flash_params& p = c.p;
        p.num_splits = splits;
        const int S = g_resolve(&p);
        if (S < 0) return raise(S, "flash_splitkv_resolve_splits");
        p.num_splits = S;  // (the launch need not work it out again)
        const int64_t rows = S > 1 ? (int64_t)p.B * p.H * S * p.Nq : 0;
        at::Tensor own;  // workspace of this call, both parts in one allocation
        if (args[4] != Py_None) {
            if (!PyTuple_CheckExact(args[4]) || PyTuple_GET_SIZE(args[4]) != 2) return not_implemented();
            const at::Tensor *wo = tensor_of(PyTuple_GET_ITEM(args[4], 0)), *wl = tensor_of(PyTuple_GET_ITEM(args[4], 1));
            for (const at::Tensor* t : {wo, wl})
                if (!t || t->scalar_type() != at::kFloat || !t->is_cuda() || !t->is_contiguous()) return not_implemented();
            if (wo->numel() < rows * p.d || wl->numel() < rows) return not_implemented();
            p.O_partial = static_cast<float*>(wo->data_ptr());
            p.LSE_partial = static_cast<float*>(wl->data_ptr());
        } else if (rows) {
            const int64_t o_floats = (rows * p.d + 63) & ~(int64_t)63;  // the second part on a 256-byte boundary
            own = empty_like_q(c, {o_floats + rows}, at::kFloat);
            p.O_partial = static_cast<float*>(own.data_ptr());
            p.LSE_partial = p.O_partial + o_floats;
        }
        if (S > 1 && (c.stream == nullptr || c.pooled_stream)) {
            p.split_counters = counters_of(c.q->device(), c.stream, c.pooled_stream);
            p.split_counters_len = p.split_counters ? fa::kCountersPerStream : 0;
        }
        return launch(g_splitkv, "flash_forward_splitkv", &c);
    });
}

// bind(addresses of flash_forward, flash_forward_splitkv, flash_splitkv_resolve_splits, FlashError): the library that
// binding.lib() has loaded
PyObject* bind(PyObject*, PyObject* args)
{
    unsigned long long f, s, r;
    PyObject* e;
    if (!PyArg_ParseTuple(args, "KKKO", &f, &s, &r, &e)) return nullptr;
    g_forward = reinterpret_cast<launch_fn>(f);
    g_splitkv = reinterpret_cast<launch_fn>(s);
    g_resolve = reinterpret_cast<resolve_fn>(r);
    Py_INCREF(e);
    Py_XSETREF(g_error, e);
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", bind, METH_VARARGS, nullptr},
    {"forward", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(forward)), METH_FASTCALL, nullptr},
    {"splitkv", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(splitkv)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void)
{
    PyObject* m = PyModule_Create(&module);
    if (m && PyModule_AddStringConstant(m, "torch_version", TORCH_VERSION) != 0) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
