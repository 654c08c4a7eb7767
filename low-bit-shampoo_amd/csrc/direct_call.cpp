// qtensor/_direct: the host side of one quantize or dequantize call of qtensor/functional.py, in native code.
//
// A call on a small matrix is bound by its host side: kernels of 4 to 6 us, and 9 us of Python around each (checks, two or
// three torch.empty, data_ptr, ctypes, the error slot).  This is the same sequence behind one call: what the tensors are is
// checked, buffers that are not given come from torch's allocator, the launch goes to torch's current stream through the
// library's entry point, the error slot is read.  Quantized and dequantized with an exact diagonal, calls back to back: 256 x 256
// 17.9 -> 12.1 us (the kernels are what is left), 1200 x 1200 17.7 -> 11.1.
//
// It takes plainly good calls only.  Anything else -- an argument that is not what it should be, a device that is not the current one, a
// tensor subclass or wrapper, a function or dispatch mode, a transformation (torch.func) or trace around the call -- returns None,
// nothing launched, and the caller's own checks say what is wrong or do it the long way: there is one place that words errors.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

namespace {

using Plain = void (*)(const void *, const void *, int, void *, void *, int, void *);
using WithDiagonal = void (*)(const void *, const void *, int, void *, void *, void *, int, void *);
// [quantize, dequantize][4, 8 bits][fp32, bf16][plain, exact diagonal]: entry points of libqtensor_hip.so (include/qtensor_hip.h)
void *entry[2][2][2][2];
int (*last_error)();
const char *(*last_error_string)();

using K = c10::DispatchKey;

// Memory of the GPU `device` and nothing around it: no wrapper that a transformation or mode has made.
bool in_plain_memory(const at::Tensor &t, int device) {
    static const c10::DispatchKeySet wrapped({K::Python, K::PythonTLSSnapshot, K::FuncTorchBatched, K::FuncTorchGradWrapper, K::Functionalize,
                                              K::Batched, K::Conjugate, K::Negative, K::ZeroTensor});
    return t.defined() && t.is_cuda() && t.layout() == at::kStrided && !t.key_set().has_any(wrapped) && t.has_storage() &&
           t.get_device() == device && t.is_contiguous();
}

// A tensor that is itself (no subclass), in plain memory of the current GPU.
const at::Tensor *plain(PyObject *obj, int device) {
    if (!THPVariable_CheckExact(obj)) return nullptr;
    const at::Tensor &t = THPVariable_Unpack(obj);
    return in_plain_memory(t, device) ? &t : nullptr;
}

// Whether something is set up around the call that would see, or wrap, the tensors it makes: with plain inputs, too, what
// at::empty returns inside a level of torch.func is a wrapper without memory of its own.
bool watched() {
    static const c10::DispatchKeySet levels({K::Python, K::PythonTLSSnapshot, K::PythonDispatcher, K::PreDispatch, K::Functionalize, K::Tracer,
                                             K::FuncTorchVmapMode, K::VmapMode, K::FuncTorchDynamicLayerFrontMode,
                                             K::FuncTorchDynamicLayerBackMode});
    return c10::impl::tls_local_dispatch_key_set().included_.has_any(levels) || at::impl::torch_function_mode_enabled();
}

// A buffer of `numel` elements: false where what is given does not fit; made if nothing is given.
bool buffer(PyObject *given, int device, long long numel, at::ScalarType type, const at::TensorOptions &like, at::Tensor &out) {
    if (given == Py_None) {
        out = at::empty({numel}, like.dtype(type));
        return in_plain_memory(out, device);
    }
    const at::Tensor *t = plain(given, device);
    if (t == nullptr || t->scalar_type() != type || t->numel() != numel) return false;
    out = *t;
    return true;
}

bool whole(PyObject *obj, long long &value) {
    if (!PyLong_CheckExact(obj)) return false;
    int overflow = 0;
    value = PyLong_AsLongLongAndOverflow(obj, &overflow);
    return overflow == 0;
}

struct Format { long long order, blocksize, bits, codes, maxima; int device; };
bool format(PyObject *data, PyObject *order, PyObject *blocksize, PyObject *bits, Format &f) {
    // (before the device is asked for: that would start the GPU's runtime for a tensor that is not there)
    if (!THPVariable_CheckExact(data) || !THPVariable_Unpack(data).is_cuda()) return false;
    if (!whole(order, f.order) || !whole(blocksize, f.blocksize) || !whole(bits, f.bits)) return false;
    if (f.bits != 4 && f.bits != 8) return false;
    if (f.blocksize < 64 || f.blocksize > 2048 || (f.blocksize & (f.blocksize - 1)) != 0) return false;
    if (f.order < 1 || f.order > 46340 || watched()) return false;
    f.codes = (f.order * f.order * f.bits + 7) / 8;
    f.maxima = f.order * ((f.order + f.blocksize - 1) / f.blocksize);
    f.device = c10::hip::current_device();
    return true;
}

const at::Tensor *code_table(PyObject *obj, const Format &f) {
    const at::Tensor *t = plain(obj, f.device);
    return t != nullptr && t->scalar_type() == at::kFloat && t->dim() == 1 && t->numel() == (1ll << f.bits) ? t : nullptr;
}

int slot_of(at::ScalarType type) { return type == at::kFloat ? 0 : type == at::kBFloat16 ? 1 : -1; }

// The launch itself, without the interpreter's lock (a full queue blocks); false with a Python error set.  Addresses first:
// asking for one may throw (a lazy copy that has to be made, memory that is not there), and nothing may between letting go
// of the lock and taking it again.
bool launch(void *fn, const at::Tensor &a, const at::Tensor &code, const Format &f, const at::Tensor &absmax, const at::Tensor *diag,
            const at::Tensor &out) {
    void *stream = c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(f.device)).stream();
    const void *from = a.data_ptr(), *table = code.data_ptr();
    void *maxima = absmax.data_ptr(), *diagonal = diag != nullptr ? diag->data_ptr() : nullptr, *to = out.data_ptr();
    const int order = (int)f.order, blocksize = (int)f.blocksize;
    const bool with_diag = diag != nullptr;
    int error = 0;
    Py_BEGIN_ALLOW_THREADS
    if (with_diag) reinterpret_cast<WithDiagonal>(fn)(from, table, order, maxima, diagonal, to, blocksize, stream);
    else reinterpret_cast<Plain>(fn)(from, table, order, maxima, to, blocksize, stream);
    error = last_error();
    Py_END_ALLOW_THREADS
    if (error == 0) return true;
    PyErr_Format(PyExc_RuntimeError, "libqtensor_hip: %s", last_error_string());
    return false;
}

// quantize(A, code, order, absmax, diag, out, blocksize, bits, with_diag) -> (out, absmax[, diag]) or None
PyObject *quantize_checked(PyObject *const *args) {
    Format f;
    if (!format(args[0], args[2], args[6], args[7], f)) Py_RETURN_NONE;
    const bool with_diag = args[8] == Py_True;
    const at::Tensor *a = plain(args[0], f.device), *code = code_table(args[1], f);
    if (a == nullptr || code == nullptr || a->numel() != f.order * f.order) Py_RETURN_NONE;
    const int slot = slot_of(a->scalar_type());
    if (slot < 0) Py_RETURN_NONE;
    const at::TensorOptions like = at::TensorOptions().device(a->device());
    at::Tensor out, absmax, diag;
    if (!buffer(args[3], f.device, f.maxima, at::kFloat, like, absmax) ||
        (with_diag && !buffer(args[4], f.device, f.order, at::kFloat, like, diag)) ||
        !buffer(args[5], f.device, f.codes, at::kByte, like, out)) Py_RETURN_NONE;
    if (!launch(entry[0][f.bits == 8][slot][with_diag], *a, *code, f, absmax, with_diag ? &diag : nullptr, out)) return nullptr;
    PyObject *result = PyTuple_New(with_diag ? 3 : 2);
    if (result == nullptr) return nullptr;
    auto put = [&](int i, PyObject *given, at::Tensor &t) {
        if (given != Py_None) Py_INCREF(given);
        PyTuple_SET_ITEM(result, i, given != Py_None ? given : THPVariable_Wrap(std::move(t)));
    };
    put(0, args[5], out);
    put(1, args[3], absmax);
    if (with_diag) put(2, args[4], diag);
    return result;
}

// dequantize(A, code, order, absmax, diag, outdtype, out, blocksize, bits, with_diag) -> out or None
PyObject *dequantize_checked(PyObject *const *args) {
    Format f;
    if (!format(args[0], args[2], args[7], args[8], f)) Py_RETURN_NONE;
    const bool with_diag = args[9] == Py_True;
    const at::Tensor *a = plain(args[0], f.device), *code = code_table(args[1], f), *absmax = plain(args[3], f.device);
    if (a == nullptr || code == nullptr || absmax == nullptr) Py_RETURN_NONE;
    if (a->scalar_type() != at::kByte || a->numel() != f.codes || absmax->scalar_type() != at::kFloat || absmax->numel() != f.maxima) Py_RETURN_NONE;
    const at::Tensor *diag = with_diag ? plain(args[4], f.device) : nullptr;
    if (with_diag && (diag == nullptr || diag->scalar_type() != at::kFloat || diag->numel() != f.order)) Py_RETURN_NONE;
    at::Tensor out;
    if (args[6] == Py_None) {
        if (!THPDtype_Check(args[5])) Py_RETURN_NONE;
        const at::ScalarType type = reinterpret_cast<THPDtype *>(args[5])->scalar_type;
        if (slot_of(type) < 0) Py_RETURN_NONE;
        out = at::empty({f.order, f.order}, at::TensorOptions().device(a->device()).dtype(type));
        if (!in_plain_memory(out, f.device)) Py_RETURN_NONE;
    } else {
        const at::Tensor *t = plain(args[6], f.device);
        if (t == nullptr || t->numel() != f.order * f.order) Py_RETURN_NONE;
        out = *t;
    }
    const int slot = slot_of(out.scalar_type());
    if (slot < 0) Py_RETURN_NONE;
    if (!launch(entry[1][f.bits == 8][slot][with_diag], *a, *code, f, *absmax, diag, out)) return nullptr;
    if (args[6] != Py_None) {
        Py_INCREF(args[6]);
        return args[6];
    }
    return THPVariable_Wrap(std::move(out));
}

// C++ exceptions (out of memory, a failed look-up) end here, with the interpreter's lock held: the caller's long way meets
// the same one and raises it in torch's words.
template <PyObject *(*body)(PyObject *const *), Py_ssize_t COUNT>
PyObject *guarded(PyObject *, PyObject *const *args, Py_ssize_t count) {
    if (count != COUNT || last_error == nullptr) Py_RETURN_NONE;
    try {
        return body(args);
    } catch (...) {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
}

// bind(addresses): the sixteen entry points in the order of `entry`, the two of the error slot
PyObject *bind(PyObject *, PyObject *list) {
    void *address[18];
    PyObject *items = PySequence_Fast(list, "bind takes a sequence of addresses");
    if (items == nullptr) return nullptr;
    if (PySequence_Fast_GET_SIZE(items) != 18) {
        Py_DECREF(items);
        PyErr_SetString(PyExc_ValueError, "bind takes eighteen addresses");
        return nullptr;
    }
    for (int i = 0; i < 18; ++i) address[i] = PyLong_AsVoidPtr(PySequence_Fast_GET_ITEM(items, i));
    Py_DECREF(items);
    if (PyErr_Occurred()) return nullptr;
    for (int i = 0; i < 18; ++i)
        if (address[i] == nullptr) {
            PyErr_SetString(PyExc_ValueError, "bind: null address");
            return nullptr;
        }
    for (int i = 0; i < 16; ++i) entry[i >> 3][(i >> 2) & 1][(i >> 1) & 1][i & 1] = address[i];
    last_error_string = reinterpret_cast<const char *(*)()>(address[17]);
    last_error = reinterpret_cast<int (*)()>(address[16]);
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", bind, METH_O, "addresses of the library's entry points"},
    {"quantize", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(guarded<quantize_checked, 9>)), METH_FASTCALL,
     "quantize(A, code, order, absmax, diag, out, blocksize, bits, with_diag): (out, absmax[, diag]), None if not taken"},
    {"dequantize", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(guarded<dequantize_checked, 10>)), METH_FASTCALL,
     "dequantize(A, code, order, absmax, diag, outdtype, out, blocksize, bits, with_diag): out, None if not taken"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_direct", "one quantize or dequantize call in native code", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// torch_version: what this was compiled against.  It reads torch's objects as they lie in memory, which no other torch promises.
PyMODINIT_FUNC PyInit__direct() {
    PyObject *made = PyModule_Create(&module);
    if (made != nullptr && PyModule_AddStringConstant(made, "torch_version", QT_TORCH_VERSION) != 0) {
        Py_DECREF(made);
        return nullptr;
    }
    return made;
}
