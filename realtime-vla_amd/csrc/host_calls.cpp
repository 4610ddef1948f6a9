// The per-observation calls of obs_transforms.py as one step each: the arguments' checks, the outputs' allocation and the launch.  A pass of three frames,
// a state and a chunk of actions is five launches of 2.5 - 2.9 us in the runtime; attribute by attribute in Python and through ctypes the same calls
// took 4.6 (frame) and 7.4 us (state, actions).  Only the plain case is taken here: exact tensors on the named device, contiguous, of the types that the kernels
// read.  For anything else a function returns None and the caller goes the general way, which converts, or reports what is wrong.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ops/empty.h>
#include <c10/hip/HIPStream.h>
#include <limits.h>
#include <string.h>
#include "../../include/rtvla.h"

namespace {

// The library's entry points as its loader found them (bind): this module is linked against none, so that there is one library in a process, whichever it is.
struct Entries {
    decltype(&rtvla_preprocess_frame) frame;
    decltype(&rtvla_preprocess_state_host) state;
    decltype(&rtvla_postprocess_actions_host) actions;
} entry;

enum { U8_HWC, F32_HWC, F32_CHW, U8_CHW };               // frame formats of rtvla_preprocess_frame

bool plain(PyObject* o) { return THPVariable_CheckExact(o); }
bool ready(const at::Tensor& t, long index) { return t.is_cuda() && t.get_device() == index && t.layout() == at::kStrided && t.is_contiguous(); }
void* stream_of(long index) { return (void*)c10::hip::getCurrentHIPStream((c10::DeviceIndex)index).stream(); }

at::Tensor like(const at::Tensor& t) { return at::empty(t.sizes(), t.options()); }

template <class F> int launch(F&& f) {                                         // (other threads run meanwhile, as behind a ctypes call)
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = f();
    Py_END_ALLOW_THREADS
    return rc;
}

// host float64 values, read before the call returns
struct Doubles {
    Py_buffer view;
    bool held = false;
    explicit Doubles(PyObject* o) {
        if (!PyObject_CheckBuffer(o)) return;
        if (PyObject_GetBuffer(o, &view, PyBUF_C_CONTIGUOUS | PyBUF_FORMAT) != 0) { PyErr_Clear(); return; }
        held = true;
    }
    ~Doubles() { if (held) PyBuffer_Release(&view); }
    bool ok() const { return held && view.itemsize == 8 && view.format && strcmp(view.format, "d") == 0 && view.len / 8 <= INT_MAX; }
    const double* data() const { return (const double*)view.buf; }
    int size() const { return (int)(view.len / 8); }
};

bool arity(Py_ssize_t got, Py_ssize_t want, const char* what) {
    if (got == want) return true;
    PyErr_Format(PyExc_TypeError, "%s takes %zd arguments (%zd given)", what, want, got);
    return false;
}

// frame(image, out_view, device index) -> status, or None
PyObject* frame(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (!arity(n, 3, "frame")) return nullptr;
    const long index = PyLong_AsLong(a[2]);
    if (index == -1 && PyErr_Occurred()) return nullptr;
    if (!entry.frame || !plain(a[0]) || !plain(a[1])) Py_RETURN_NONE;
    const at::Tensor& img = THPVariable_Unpack(a[0]);
    const at::Tensor& out = THPVariable_Unpack(a[1]);
    const bool f32 = img.scalar_type() == at::kFloat;
    if ((!f32 && img.scalar_type() != at::kByte) || img.dim() != 3 || !ready(img, index)) Py_RETURN_NONE;
    if (out.scalar_type() != at::kBFloat16 || out.dim() != 3 || out.size(0) != 224 || out.size(1) != 224 || out.size(2) != 3 || !ready(out, index)) Py_RETURN_NONE;
    const bool chw = img.size(0) == 3;
    const int64_t h = img.size(chw ? 1 : 0), w = img.size(chw ? 2 : 1);
    if ((!chw && img.size(2) != 3) || h > INT_MAX || w > INT_MAX) Py_RETURN_NONE;
    const int format = f32 ? (chw ? F32_CHW : F32_HWC) : (chw ? U8_CHW : U8_HWC);
    void* const src = img.data_ptr();
    void* const dst = out.data_ptr();
    void* const stream = stream_of(index);
    return PyLong_FromLong(launch([&] { return entry.frame(src, format, (int)h, (int)w, dst, stream); }));
    END_HANDLE_TH_ERRORS
}

// state(values, stat_a, stat_b, number of statistics, mode, like z, like the bins or None, bf16 output or None, device index) -> (z, bins), status or None
PyObject* state(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (!arity(n, 9, "state")) return nullptr;
    const long n_stats = PyLong_AsLong(a[3]), mode = PyLong_AsLong(a[4]), index = PyLong_AsLong(a[8]);
    if (PyErr_Occurred()) return nullptr;
    if (!entry.state || !plain(a[1]) || !plain(a[2]) || !plain(a[5]) || (a[6] != Py_None && !plain(a[6])) || (a[7] != Py_None && !plain(a[7]))) Py_RETURN_NONE;
    if (a[7] != Py_None) {
        const at::Tensor& t = THPVariable_Unpack(a[7]);
        if (t.scalar_type() != at::kBFloat16 || !ready(t, index) || t.numel() < 32) Py_RETURN_NONE;
    }
    Doubles values(a[0]);
    if (!values.ok()) Py_RETURN_NONE;
    const at::Tensor z = like(THPVariable_Unpack(a[5]));
    at::Tensor bins;
    if (a[6] != Py_None) bins = like(THPVariable_Unpack(a[6]));
    const double* const sa = (const double*)THPVariable_Unpack(a[1]).data_ptr();
    const double* const sb = (const double*)THPVariable_Unpack(a[2]).data_ptr();
    void* const bf16 = a[7] != Py_None ? THPVariable_Unpack(a[7]).data_ptr() : nullptr;
    double* const zp = (double*)z.data_ptr();
    int32_t* const bp = bins.defined() ? (int32_t*)bins.data_ptr() : nullptr;
    void* const stream = stream_of(index);
    const int rc = launch([&] { return entry.state(values.data(), values.size(), sa, sb, (int)n_stats, (int)mode, bf16, zp, bp, stream); });
    if (rc) return PyLong_FromLong(rc);
    PyObject* const result = PyTuple_New(2);
    if (!result) return nullptr;
    PyTuple_SET_ITEM(result, 0, THPVariable_Wrap(z));
    if (bins.defined()) PyTuple_SET_ITEM(result, 1, THPVariable_Wrap(bins));
    else { Py_INCREF(Py_None); PyTuple_SET_ITEM(result, 1, Py_None); }
    return result;
    END_HANDLE_TH_ERRORS
}

// actions(actions, values, stat_a, stat_b, number of statistics, mode, action_dim, like a row of the result, device index) -> result, status or None
PyObject* actions(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (!arity(n, 9, "actions")) return nullptr;
    const long n_stats = PyLong_AsLong(a[4]), mode = PyLong_AsLong(a[5]), dim = PyLong_AsLong(a[6]), index = PyLong_AsLong(a[8]);
    if (PyErr_Occurred()) return nullptr;
    if (!entry.actions || !plain(a[0]) || !plain(a[2]) || !plain(a[3]) || !plain(a[7])) Py_RETURN_NONE;
    const at::Tensor& act = THPVariable_Unpack(a[0]);
    if (act.scalar_type() != at::kBFloat16 || act.dim() != 2 || act.size(1) != 32 || !ready(act, index) || act.size(0) > INT_MAX || dim < 0) Py_RETURN_NONE;
    Doubles values(a[1]);
    if (!values.ok()) Py_RETURN_NONE;
    const at::Tensor out = at::empty({act.size(0), dim}, THPVariable_Unpack(a[7]).options());
    void* const src = act.data_ptr();
    const double* const sa = (const double*)THPVariable_Unpack(a[2]).data_ptr();
    const double* const sb = (const double*)THPVariable_Unpack(a[3]).data_ptr();
    double* const dst = (double*)out.data_ptr();
    void* const stream = stream_of(index);
    const int rc = launch([&] {
        return entry.actions(src, (int)act.size(0), sa, sb, (int)n_stats, (int)mode, values.data(), values.size(), (int)dim, dst, stream);
    });
    return rc ? PyLong_FromLong(rc) : THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

// bind(address of rtvla_preprocess_frame, of rtvla_preprocess_state_host, of rtvla_postprocess_actions_host): once, before any other call
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (!arity(n, 3, "bind")) return nullptr;
    void* const at[3] = {PyLong_AsVoidPtr(a[0]), PyLong_AsVoidPtr(a[1]), PyLong_AsVoidPtr(a[2])};
    if (PyErr_Occurred()) return nullptr;
    entry = {(decltype(entry.frame))at[0], (decltype(entry.state))at[1], (decltype(entry.actions))at[2]};
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {{"bind", (PyCFunction)(void*)bind, METH_FASTCALL, nullptr},
                         {"frame", (PyCFunction)(void*)frame, METH_FASTCALL, nullptr},
                         {"state", (PyCFunction)(void*)state, METH_FASTCALL, nullptr},
                         {"actions", (PyCFunction)(void*)actions, METH_FASTCALL, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_rtvla_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__rtvla_host(void) { return PyModule_Create(&module); }
