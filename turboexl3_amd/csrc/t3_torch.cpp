// The Python entry points' way into the C ABI: reads torch tensors, allocates the output, finds the thread's workspace and
// calls the library, all in one native call.
//
// Why it is native: a decode-row call's kernels take 7 to 14 us, and building the same descriptors field by field from
// Python took 14 us a dense call and 24 to 36 us a routed one (a bank is nine arrays), so the host and not the GPU set the
// pace of a decode loop. Nothing is kept between calls but the interned attribute names and each thread's workspace
// key: every call reads its own tensors.

#include <Python.h>

#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <optional>

#include "../../include/turboexl3_hip.h"

namespace {

PyObject* g_workspaces = nullptr;  // api._workspaces: {(device type, device index, thread): uint8 tensor}
PyObject* g_workspace = nullptr;   // api._workspace(device, bytes): makes or grows the thread's entry
PyObject* g_error = nullptr;       // api.T3Error
PyObject *s_codebook, *s_window, *s_gate, *s_up, *s_down, *s_trellis, *s_suh, *s_svh, *s_cuda_stream, *s_device, *s_cuda;

// Thrown where a Python exception is already set.
struct PythonError {};

[[noreturn]] void refuse(int32_t status) {
    PyObject* v = PyLong_FromLong(status);
    PyErr_SetObject(g_error, v);
    Py_XDECREF(v);
    throw PythonError{};
}
void check(int32_t status) {
    if (status != T3_OK) refuse(status);
}

// A tensor's descriptor, and the tensor that owns its bytes (a contiguous copy where the caller's is not). It is held until
// the call is over whoever else holds it: an attribute may be computed and have no other owner, and another thread may
// replace a bank's while this one runs without the interpreter lock; memory freed meanwhile would be handed out again as
// the call's own output or workspace.
struct Arg {
    t3_array a;
    at::Tensor keep;
};

int32_t dtype_of(at::ScalarType t) {
    switch (t) {
        case at::kFloat: return T3_F32;
        case at::kHalf: return T3_F16;
        case at::kBFloat16: return T3_BF16;
        case at::kUInt16: return T3_U16;
        case at::kShort: return T3_I16;
        case at::kUInt32: return T3_U32;
        case at::kInt: return T3_I32;
        default: return -1;
    }
}

void describe(const at::TensorBase& t, int32_t dtype, t3_array* a) {
    a->data = t.data_ptr();
    a->ndim = static_cast<int32_t>(t.dim());
    a->dtype = dtype;
    const auto shape = t.sizes();
    for (size_t i = 0; i < shape.size(); ++i) a->shape[i] = shape[i];
}

void read(PyObject* o, Arg* out) {
    if (!THPVariable_Check(o)) {
        PyErr_SetString(PyExc_TypeError, "expected a torch.Tensor");
        throw PythonError{};
    }
    const at::Tensor& t = THPVariable_Unpack(o);
    const int32_t dtype = dtype_of(t.scalar_type());
    if (dtype < 0) refuse(T3_BadExl3Dtype);
    if (t.dim() > T3_MAX_DIMS) refuse(T3_BadExl3Shape);
    if (!t.is_cuda()) {
        PyErr_SetString(PyExc_ValueError, "turboexl3_amd runs on device tensors only");
        throw PythonError{};
    }
    out->keep = t.is_contiguous() ? t : t.contiguous();
    describe(out->keep, dtype, &out->a);
}

// An attribute of a Python object, owned for the scope.
struct Attr {
    PyObject* p;
    Attr(PyObject* o, PyObject* name) : p(PyObject_GetAttr(o, name)) {
        if (!p) throw PythonError{};
    }
    ~Attr() { Py_DECREF(p); }
    Attr(const Attr&) = delete;
};

long as_long(PyObject* o) {
    const long v = PyLong_AsLong(o);
    if (v == -1 && PyErr_Occurred()) throw PythonError{};
    return v;
}

t3_decode read_decode(PyObject* o) {
    const Attr cb(o, s_codebook), wb(o, s_window);
    return t3_decode{static_cast<int32_t>(as_long(cb.p)), static_cast<int32_t>(as_long(wb.p))};
}

struct BankArg {
    t3_bank b;
    at::Tensor keep[9];
};

void read_proj(PyObject* bank, PyObject* name, t3_proj* p, at::Tensor* keep) {
    const Attr proj(bank, name);
    PyObject* const names[3] = {s_trellis, s_suh, s_svh};
    t3_array* const arrays[3] = {&p->trellis, &p->suh, &p->svh};
    for (int i = 0; i < 3; ++i) {
        const Attr t(proj.p, names[i]);
        Arg a;
        read(t.p, &a);
        *arrays[i] = a.a;
        keep[i] = std::move(a.keep);
    }
}

void read_bank(PyObject* o, BankArg* out) {
    read_proj(o, s_gate, &out->b.gate, out->keep);
    read_proj(o, s_up, &out->b.up, out->keep + 3);
    read_proj(o, s_down, &out->b.down, out->keep + 6);
}

// The stream a call runs on: the caller's, or the current one. A given stream is the current one of x's device for the
// scope, so that whatever the call makes on the way, the contiguous copies, the output and a workspace that is cleared, is
// made in that stream's order and not beside it.
class CallStream {
public:
    CallStream(PyObject* stream, PyObject* x) {
        if (stream == Py_None) return;
        const Attr s(stream, s_cuda_stream);
        void* p = PyLong_AsVoidPtr(s.p);
        if (!p && PyErr_Occurred()) throw PythonError{};
        given_ = true;
        raw_ = p;
        if (!THPVariable_Check(x) || !THPVariable_Unpack(x).is_cuda()) return;  // read() refuses it
        const c10::DeviceIndex device = THPVariable_Unpack(x).device().index();
        const c10::hip::HIPStream now = c10::hip::getCurrentHIPStream(device);
        if (now.stream() == static_cast<hipStream_t>(p)) return;
        before_ = now;
        c10::hip::setCurrentHIPStream(c10::hip::getStreamFromExternal(static_cast<hipStream_t>(p), device));
    }
    ~CallStream() {
        if (before_) c10::hip::setCurrentHIPStream(*before_);
    }
    CallStream(const CallStream&) = delete;
    t3_stream get() const { return given_ ? raw_ : c10::hip::getCurrentHIPStream().stream(); }

private:
    bool given_ = false;
    void* raw_ = nullptr;
    std::optional<c10::hip::HIPStream> before_;
};

struct Workspace {
    at::Tensor keep;
    void* p;
    size_t bytes;
    explicit Workspace(const at::Tensor& t) : keep(t), p(t.data_ptr()), bytes(static_cast<size_t>(t.numel())) {}
};

// The thread's workspace on x's device, grown by the Python side where it is too small. The dict owns it and stays the
// one place that says which it is; this side keeps only the key of a thread's last device.
Workspace workspace_for(PyObject* x, size_t need) {
    static thread_local PyObject* key = nullptr;
    static thread_local int key_device = -1;
    const int device = THPVariable_Unpack(x).device().index();
    if (key_device != device) {
        Py_XDECREF(key);
        key_device = -1;
        key = Py_BuildValue("(OiN)", s_cuda, device, PyLong_FromUnsignedLong(PyThread_get_thread_ident()));
        if (!key) throw PythonError{};
        key_device = device;
    }
    PyObject* ws = PyDict_GetItemWithError(g_workspaces, key);
    if (!ws && PyErr_Occurred()) throw PythonError{};
    if (ws) {
        const at::Tensor& t = THPVariable_Unpack(ws);
        if (static_cast<size_t>(t.numel()) >= need) return Workspace(t);
    }
    const Attr dev(x, s_device);
    PyObject* made = PyObject_CallFunction(g_workspace, "On", dev.p, static_cast<Py_ssize_t>(need));
    if (!made) throw PythonError{};
    const Workspace w(THPVariable_Unpack(made));
    Py_DECREF(made);
    return w;
}

// A new contiguous tensor of x's dtype and device, x's shape with the last width replaced (width < 0: as it is).
at::TensorBase new_output(PyObject* xo, int64_t width, t3_array* ay) {
    const at::Tensor& x = THPVariable_Unpack(xo);
    int64_t shape[T3_MAX_DIMS];
    const size_t nd = static_cast<size_t>(x.dim());
    for (size_t i = 0; i < nd; ++i) shape[i] = x.size(static_cast<int64_t>(i));
    if (width >= 0 && nd > 0) shape[nd - 1] = width;
    at::TensorBase y = at::detail::empty_cuda(at::IntArrayRef(shape, nd), x.scalar_type(), x.device(), std::nullopt);
    describe(y, dtype_of(x.scalar_type()), ay);
    return y;
}

// Runs f, which returns a new tensor, with C++ and library failures as Python exceptions.
template <typename F>
PyObject* guarded(F&& f) {
    try {
        return THPVariable_Wrap(f());
    } catch (const PythonError&) {
        return nullptr;
    } catch (...) {
        torch::translate_exception_to_python(std::current_exception());
        return nullptr;
    }
}

bool arity(Py_ssize_t got, Py_ssize_t want) {
    if (got == want) return true;
    PyErr_Format(PyExc_TypeError, "%zd arguments where %zd are taken", got, want);
    return false;
}

// The library's calls run without the interpreter lock, so that another thread's Python goes on meanwhile.
template <typename F>
void unlocked(F&& f) {
    int32_t st;
    Py_BEGIN_ALLOW_THREADS
    st = f();
    Py_END_ALLOW_THREADS
    check(st);
}

// linear(x, trellis, suh, svh, bias or None, dec, stream, chain)
PyObject* py_linear(PyObject*, PyObject* const* v, Py_ssize_t n) {
    if (!arity(n, 8)) return nullptr;
    return guarded([&] {
        const CallStream on(v[6], v[0]);
        Arg x, t, suh, svh, bias;
        read(v[0], &x);
        read(v[1], &t);
        read(v[2], &suh);
        read(v[3], &svh);
        const bool has_bias = v[4] != Py_None;
        if (has_bias) read(v[4], &bias);
        const t3_decode dec = read_decode(v[5]);
        size_t need = 0;
        check(t3_linear_workspace_bytes(&x.a, &t.a, dec, &need));
        const t3_stream stream = on.get();
        const bool chain = v[7] == Py_True;
        t3_array ay;
        at::TensorBase y = new_output(v[0], t.a.shape[1] * 16, &ay);
        const Workspace ws = workspace_for(v[0], need);
        unlocked([&] {
            if (has_bias) return t3_linear_bias(stream, &x.a, &t.a, &suh.a, &svh.a, &bias.a, dec, &ay, ws.p, ws.bytes);
            return (chain ? t3_linear_chain : t3_linear)(stream, &x.a, &t.a, &suh.a, &svh.a, dec, &ay, ws.p, ws.bytes);
        });
        return y;
    });
}

// linear_resident(x, w_hat, suh, svh, stream)
PyObject* py_linear_resident(PyObject*, PyObject* const* v, Py_ssize_t n) {
    if (!arity(n, 5)) return nullptr;
    return guarded([&] {
        const CallStream on(v[4], v[0]);
        Arg x, w, suh, svh;
        read(v[0], &x);
        read(v[1], &w);
        read(v[2], &suh);
        read(v[3], &svh);
        size_t need = 0;
        check(t3_linear_resident_workspace_bytes(&x.a, &w.a, &need));
        const t3_stream stream = on.get();
        t3_array ay;
        at::TensorBase y = new_output(v[0], w.a.shape[1], &ay);
        const Workspace ws = workspace_for(v[0], need);
        unlocked([&] { return t3_linear_resident(stream, &x.a, &w.a, &suh.a, &svh.a, &ay, ws.p, ws.bytes); });
        return y;
    });
}

// linear_unrot(x, w_std, col0, cols, stream, parts)
PyObject* py_linear_unrot(PyObject*, PyObject* const* v, Py_ssize_t n) {
    if (!arity(n, 6)) return nullptr;
    return guarded([&] {
        const CallStream on(v[4], v[0]);
        Arg x, w;
        read(v[0], &x);
        read(v[1], &w);
        const int64_t col0 = as_long(v[2]), cols = as_long(v[3]);
        if (cols < 0) refuse(T3_BadExl3Shape);
        const t3_stream stream = on.get();
        size_t need = 0;
        if (v[5] == Py_True) check(t3_linear_unrot_workspace_bytes(&x.a, &w.a, col0, cols, &need));
        t3_array ay;
        at::TensorBase y = new_output(v[0], cols, &ay);
        if (v[5] == Py_True) {
            const Workspace ws = workspace_for(v[0], need);
            unlocked([&] { return t3_linear_unrot_parts(stream, &x.a, &w.a, col0, cols, &ay, ws.p, ws.bytes); });
        } else {
            unlocked([&] { return t3_linear_unrot(stream, &x.a, &w.a, col0, cols, &ay); });
        }
        return y;
    });
}

enum MoeEntry : long { kMoe, kClamped, kSwiglu, kWithShared, kSharedExpert };

// moe(entry, x, bank, inds, scores, dec, limit or verify_rows, clamp_at, shared tensor / bank / None, stream)
PyObject* py_moe(PyObject*, PyObject* const* v, Py_ssize_t n) {
    if (!arity(n, 10)) return nullptr;
    return guarded([&] {
        const CallStream on(v[9], v[1]);
        const long entry = as_long(v[0]);
        Arg x, inds, scores, add;
        BankArg bank, shared;
        read(v[1], &x);
        read(v[3], &inds);
        read(v[4], &scores);
        read_bank(v[2], &bank);
        if (entry == kWithShared) read(v[8], &add);
        if (entry == kSharedExpert) read_bank(v[8], &shared);
        const t3_decode dec = read_decode(v[5]);
        const int32_t i0 = static_cast<int32_t>(as_long(v[6])), i1 = static_cast<int32_t>(as_long(v[7]));
        size_t need = 0;
        check(t3_moe_workspace_bytes(&x.a, &bank.b, &inds.a, entry == kSharedExpert ? &shared.b : nullptr, &need));
        const t3_stream stream = on.get();
        t3_array ay;
        at::TensorBase y = new_output(v[1], -1, &ay);
        const Workspace ws = workspace_for(v[1], need);
        unlocked([&] {
            switch (entry) {
                case kClamped:
                    return t3_moe_clamped(stream, &x.a, &bank.b, &inds.a, &scores.a, dec, i0, &ay, ws.p, ws.bytes);
                case kSwiglu:
                    return t3_moe_swiglu(stream, &x.a, &bank.b, &inds.a, &scores.a, dec, i0, i1, &ay, ws.p, ws.bytes);
                case kWithShared:
                    return t3_moe_with_shared(stream, &x.a, &bank.b, &inds.a, &scores.a, dec, i0, &add.a, &ay, ws.p,
                                              ws.bytes);
                case kSharedExpert:
                    return t3_moe_shared_expert(stream, &x.a, &bank.b, &inds.a, &scores.a, dec, i0, &shared.b, &ay, ws.p,
                                                ws.bytes);
                default: return t3_moe(stream, &x.a, &bank.b, &inds.a, &scores.a, dec, i0, &ay, ws.p, ws.bytes);
            }
        });
        return y;
    });
}

// moe_fused_shared(x, bank, inds, scores, dec, shared bank, sigtab, logit, stream)
PyObject* py_moe_fused_shared(PyObject*, PyObject* const* v, Py_ssize_t n) {
    if (!arity(n, 9)) return nullptr;
    return guarded([&] {
        const CallStream on(v[8], v[0]);
        Arg x, inds, scores, tab, logit;
        BankArg bank, shared;
        read(v[0], &x);
        read(v[2], &inds);
        read(v[3], &scores);
        read_bank(v[1], &bank);
        read_bank(v[5], &shared);
        const t3_decode dec = read_decode(v[4]);
        size_t need = 0;
        check(t3_moe_workspace_bytes(&x.a, &bank.b, &inds.a, &shared.b, &need));
        read(v[6], &tab);
        read(v[7], &logit);
        const t3_stream stream = on.get();
        t3_array ay;
        at::TensorBase y = new_output(v[0], -1, &ay);
        const Workspace ws = workspace_for(v[0], need);
        unlocked([&] {
            return t3_moe_fused_shared(stream, &x.a, &bank.b, &inds.a, &scores.a, dec, &shared.b, &tab.a, &logit.a, &ay,
                                       ws.p, ws.bytes);
        });
        return y;
    });
}

// moe_fused_shared_routed(x, bank, logits, k, dec, shared bank, sigtab, logit or None, gate_vec or None, stream)
PyObject* py_moe_fused_shared_routed(PyObject*, PyObject* const* v, Py_ssize_t n) {
    if (!arity(n, 10)) return nullptr;
    return guarded([&] {
        const CallStream on(v[9], v[0]);
        Arg x, logits, tab, logit, gate;
        BankArg bank, shared;
        read(v[0], &x);
        read(v[2], &logits);
        read_bank(v[1], &bank);
        read_bank(v[5], &shared);
        const int64_t k = as_long(v[3]);
        const t3_decode dec = read_decode(v[4]);
        size_t need = 0;
        check(t3_moe_fused_shared_routed_workspace_bytes(&x.a, &bank.b, &logits.a, k, &shared.b, &need));
        read(v[6], &tab);
        if (v[7] != Py_None) read(v[7], &logit);
        if (v[8] != Py_None) read(v[8], &gate);
        const t3_stream stream = on.get();
        t3_array ay;
        at::TensorBase y = new_output(v[0], -1, &ay);
        const Workspace ws = workspace_for(v[0], need);
        unlocked([&] {
            return t3_moe_fused_shared_routed(stream, &x.a, &bank.b, &logits.a, k, dec, &shared.b, &tab.a,
                                              v[7] != Py_None ? &logit.a : nullptr, v[8] != Py_None ? &gate.a : nullptr, &ay,
                                              ws.p, ws.bytes);
        });
        return y;
    });
}

// bind(workspaces dict, workspace function, error class): once, when turboexl3_amd.api is imported
PyObject* py_bind(PyObject*, PyObject* const* v, Py_ssize_t n) {
    if (!arity(n, 3)) return nullptr;
    PyObject** const to[3] = {&g_workspaces, &g_workspace, &g_error};
    for (int i = 0; i < 3; ++i) {
        Py_INCREF(v[i]);
        Py_XSETREF(*to[i], v[i]);
    }
    Py_RETURN_NONE;
}

#define T3_METHOD(name, f) {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(f)), METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {
    T3_METHOD("bind", py_bind),
    T3_METHOD("linear", py_linear),
    T3_METHOD("linear_resident", py_linear_resident),
    T3_METHOD("linear_unrot", py_linear_unrot),
    T3_METHOD("moe", py_moe),
    T3_METHOD("moe_fused_shared", py_moe_fused_shared),
    T3_METHOD("moe_fused_shared_routed", py_moe_fused_shared_routed),
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_t3_torch", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__t3_torch() {
    struct {
        PyObject** at;
        const char* text;
    } const names[] = {{&s_codebook, "codebook"}, {&s_window, "window_bits"}, {&s_gate, "gate"}, {&s_up, "up"},
                       {&s_down, "down"}, {&s_trellis, "trellis"}, {&s_suh, "suh"}, {&s_svh, "svh"},
                       {&s_cuda_stream, "cuda_stream"}, {&s_device, "device"}, {&s_cuda, "cuda"}};
    for (const auto& name : names)
        if (!(*name.at = PyUnicode_InternFromString(name.text))) return nullptr;
    return PyModule_Create(&kModule);
}
