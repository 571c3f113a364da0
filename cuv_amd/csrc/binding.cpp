// The Python calls' way into libcuvdia.so: checks the operands as cuv_amd/dia.py does and calls the C ABI.
//
// A call from Python through ctypes spends about 8 us on the host -- attribute and stride look-ups, a device context,
// the stream, argument conversion --, more than the kernels of a small layer take.  Here the same steps read the
// tensors' fields directly (under 1 us).  Every function returns True when it has done the call, and False -- having
// done nothing -- for operands that are not the usual ones (wrong shapes or types, another device, a matrix without
// a descriptor yet, a capturing stream, a tensor without memory of its own): dia.py then takes its general way, which also words the errors.  Once the
// library has been called a failure is raised, as _lib.CuvDiaError: kernels may be queued, and the general way would
// do the call a second time.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>
#include <torch/version.h>

#include <cctype>
#include <cstring>
#include <string>

#include "cuvdia.h"

namespace {

struct Names {
    PyObject *h, *w, *vec, *desc;
} g_names;

// One operand as a column-major matrix: tensor of shape (batch, rows).
struct Dense {
    float *p = nullptr;
    long long ld = 0, rows = 0, batch = 0;
    int device = -1;
};

bool float_tensor(PyObject *o, const at::Tensor *&t)
{
    if (!THPVariable_Check(o)) return false;
    t = &THPVariable_Unpack(o);
    return t->has_storage() && t->is_cuda() && t->scalar_type() == at::kFloat && t->layout() == at::kStrided;
}

bool dense(PyObject *o, Dense &d)
{
    const at::Tensor *t;
    if (!float_tensor(o, t) || t->dim() != 2 || t->stride(1) != 1) return false;
    d.batch = t->size(0);
    d.rows = t->size(1);
    d.ld = d.batch > 1 ? t->stride(0) : d.rows;
    d.device = t->get_device();
    d.p = static_cast<float *>(t->data_ptr());
    return d.p && d.batch > 0 && d.batch <= 0x7fffffff && d.rows > 0 && d.ld >= d.rows;
}

struct Matrix {
    const cuvdia_desc *desc = nullptr;
    float *vals = nullptr;
    long long h = 0, w = 0;
    int device = -1;
};

bool read_int(PyObject *o, PyObject *name, long long &v)
{
    PyObject *a = PyObject_GetAttr(o, name);
    if (!a) { PyErr_Clear(); return false; }
    const bool ok = PyLong_CheckExact(a);
    if (ok) v = PyLong_AsLongLong(a);
    Py_DECREF(a);
    if (PyErr_Occurred()) { PyErr_Clear(); return false; }
    return ok;
}

bool matrix(PyObject *o, Matrix &m)
{
    long long desc = 0;
    if (!read_int(o, g_names.desc, desc) || desc == 0 || !read_int(o, g_names.h, m.h) || !read_int(o, g_names.w, m.w)) return false;
    m.desc = reinterpret_cast<const cuvdia_desc *>(desc);
    THPObjectPtr vec(PyObject_GetAttr(o, g_names.vec));      // (the matrix holds it)
    if (!vec) { PyErr_Clear(); return false; }
    const at::Tensor *t;
    if (!float_tensor(vec.get(), t)) return false;
    m.vals = static_cast<float *>(t->data_ptr());
    m.device = t->get_device();
    return m.vals != nullptr;
}

// Whether a runtime call succeeded; takes its error from the runtime, where the general way's launch would find it.
bool ok(hipError_t e)
{
    if (e != hipSuccess) (void)hipGetLastError();
    return e == hipSuccess;
}

// The stream to launch on; false when `device` is not the current one or -- for a call that waits -- is being captured
// (or cannot be asked: the default stream while another thread captures).
bool stream_of(int device, bool sync, hipStream_t &s)
{
    int current = -1;
    if (!ok(hipGetDevice(&current)) || current != device) return false;
    s = c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(device)).stream();
    if (sync) {
        hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
        if (!ok(hipStreamIsCapturing(s, &status)) || status != hipStreamCaptureStatusNone) return false;
    }
    return true;
}

PyObject *no() { Py_RETURN_FALSE; }

// Raises _lib.CuvDiaError(code, what); returns nullptr.
PyObject *raise(int code, const char *what)
{
    PyObject *lib = PyImport_ImportModule("cuv_amd._lib");
    PyObject *type = lib ? PyObject_GetAttrString(lib, "CuvDiaError") : nullptr;
    PyObject *error = type ? PyObject_CallFunction(type, "is", code, what) : nullptr;
    if (error) PyErr_SetObject(type, error);
    Py_XDECREF(error);
    Py_XDECREF(type);
    Py_XDECREF(lib);
    return nullptr;
}

// Runs call(), named `what`, and, if asked to, waits for it, both without holding the interpreter: a launch, too, blocks
// where the stream's queue is full.
template <class Call>
PyObject *run(bool sync, hipStream_t s, const char *what, Call &&call)
{
    if (sync && cuvdia_wait_begin() != CUVDIA_OK) return no();
    int rc = CUVDIA_OK, waited = CUVDIA_OK;
    Py_BEGIN_ALLOW_THREADS
    rc = call();
    if (sync) waited = cuvdia_wait_end(s);
    Py_END_ALLOW_THREADS
    if (rc != CUVDIA_OK) return raise(rc, what);
    if (waited != CUVDIA_OK) return raise(waited, "cuvdia_wait_end");
    Py_RETURN_TRUE;
}

// 'n' or 't' from a one-character string, 0 otherwise
char trans_of(PyObject *o)
{
    if (!PyUnicode_CheckExact(o) || PyUnicode_GetLength(o) != 1) return 0;
    const Py_UCS4 c = PyUnicode_READ_CHAR(o, 0);
    return c == 'n' || c == 't' ? (char)c : 0;
}

bool number(PyObject *o, float &v)
{
    if (!PyFloat_CheckExact(o) && !PyLong_CheckExact(o)) return false;
    v = static_cast<float>(PyFloat_AsDouble(o));
    if (PyErr_Occurred()) { PyErr_Clear(); return false; }
    return true;
}

// product(dst, A, B, transA, factAB, factC, bias, act, seed, sync)
PyObject *product(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    Dense dst, B;
    Matrix A;
    float alpha, beta;
    if (n != 10 || !dense(a[0], dst) || !matrix(a[1], A) || !dense(a[2], B) || !number(a[4], alpha) || !number(a[5], beta)) return no();
    const char trans = trans_of(a[3]);
    const long long n_out = trans == 't' ? A.w : A.h, n_in = trans == 't' ? A.h : A.w;
    if (!trans || dst.rows != n_out || B.rows != n_in || dst.batch != B.batch || A.device != dst.device || B.device != dst.device) return no();
    const float *bias = nullptr;
    if (a[6] != Py_None) {
        const at::Tensor *t;
        if (!float_tensor(a[6], t) || !t->is_contiguous() || t->numel() != n_out || t->get_device() != dst.device) return no();
        bias = static_cast<const float *>(t->data_ptr());
        if (!bias) return no();
    }
    if (!PyLong_CheckExact(a[7]) || !PyLong_CheckExact(a[8])) return no();
    const int act = (int)PyLong_AsLong(a[7]);
    const unsigned long long seed = PyLong_AsUnsignedLongLongMask(a[8]);
    if (PyErr_Occurred()) { PyErr_Clear(); return no(); }
    const bool sync = PyObject_IsTrue(a[9]) == 1;
    hipStream_t s;
    if (!stream_of(dst.device, sync, s)) return no();
    return run(sync, s, "cuvdia_spmm_layer_f32", [&] {
        return cuvdia_spmm_layer_f32(A.desc, A.vals, B.p, B.ld, dst.p, dst.ld, (int)B.batch, trans, alpha, beta, bias, act, seed, s);
    });
}

// projection(C, A, B, factAB, factC, sync)
PyObject *projection(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    Matrix C;
    Dense A, B;
    float alpha, beta;
    if (n != 6 || !matrix(a[0], C) || !dense(a[1], A) || !dense(a[2], B) || !number(a[3], alpha) || !number(a[4], beta)) return no();
    if (A.rows != C.h || B.rows != C.w || A.batch != B.batch || A.device != C.device || B.device != C.device) return no();
    const bool sync = PyObject_IsTrue(a[5]) == 1;
    hipStream_t s;
    if (!stream_of(C.device, sync, s)) return no();
    return run(sync, s, "cuvdia_dd2dia_f32", [&] {
        return cuvdia_dd2dia_f32(C.desc, C.vals, A.p, A.ld, B.p, B.ld, (int)A.batch, alpha, beta, s);
    });
}

// weight_step(w, m or None, dw, learnrate, momentum_weight, decay, sync): the value vectors themselves
PyObject *weight_step(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    if (n != 7) return no();
    const at::Tensor *w, *d, *m = nullptr;
    if (!float_tensor(a[0], w) || !float_tensor(a[2], d) || !w->is_contiguous() || !d->is_contiguous()) return no();
    if (a[1] != Py_None && (!float_tensor(a[1], m) || !m->is_contiguous())) return no();
    const long long count = w->numel();
    float lr, mw, decay;
    if (count < 1 || d->numel() != count || (m && m->numel() != count) || !number(a[3], lr) || !number(a[4], mw) || !number(a[5], decay)) return no();
    const int device = w->get_device();
    if (d->get_device() != device || (m && m->get_device() != device)) return no();
    const bool sync = PyObject_IsTrue(a[6]) == 1;
    hipStream_t s;
    if (!stream_of(device, sync, s)) return no();
    float *wp = static_cast<float *>(w->data_ptr());
    const float *dp = static_cast<const float *>(d->data_ptr());
    float *mp = m ? static_cast<float *>(m->data_ptr()) : nullptr;
    if (!wp || !dp || (m && !mp)) return no();
    return run(sync, s, mp ? "cuvdia_learn_step_weight_decay_momentum_f32" : "cuvdia_learn_step_weight_decay_f32", [&] {
        return mp ? cuvdia_learn_step_weight_decay_momentum_f32(wp, mp, dp, count, lr, mw, decay, s)
                 : cuvdia_learn_step_weight_decay_f32(wp, dp, count, lr, decay, s);
    });
}

// The functions as Python calls them.  Reading a tensor's fields throws where there are none to read (a wrapper seen
// inside a transform, a fake tensor); the library's own calls, which come last, do not throw.
template <PyObject *(*Function)(PyObject *, PyObject *const *, Py_ssize_t)>
PyObject *guarded(PyObject *self, PyObject *const *a, Py_ssize_t n)
{
    try {
        return Function(self, a, n);
    } catch (const std::exception &) {
        PyErr_Clear();
        return no();
    }
}

template <PyObject *(*Function)(PyObject *, PyObject *const *, Py_ssize_t)>
PyMethodDef method(const char *name)
{
    return {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(guarded<Function>)), METH_FASTCALL, nullptr};
}
PyMethodDef g_methods[] = {method<product>("product"), method<projection>("projection"), method<weight_step>("weight_step"),
                           {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_native", "Direct calls into libcuvdia.so.", -1, g_methods, nullptr, nullptr, nullptr, nullptr};

// Fails to import where torch or Python is not the one this was compiled against: a tensor's fields may lie elsewhere.
bool fits()
{
    PyObject *torch = PyImport_ImportModule("torch");
    PyObject *version = torch ? PyObject_GetAttrString(torch, "__version__") : nullptr;
    const char *text = version ? PyUnicode_AsUTF8(version) : nullptr;
    const size_t n = std::strlen(TORCH_VERSION);                   // (what follows names the build: "+rocm7.0")
    const bool same_torch = text && std::strncmp(text, TORCH_VERSION, n) == 0 && !std::isdigit((unsigned char)text[n]);
    const std::string python = std::to_string(PY_MAJOR_VERSION) + "." + std::to_string(PY_MINOR_VERSION) + ".";
    const bool same_python = std::strncmp(Py_GetVersion(), python.c_str(), python.size()) == 0;
    if (!PyErr_Occurred() && !(same_torch && same_python))
        PyErr_Format(PyExc_ImportError, "built for torch %s and Python %sx, this is torch %s and Python %s", TORCH_VERSION, python.c_str(), text ? text : "?", Py_GetVersion());
    Py_XDECREF(version);
    Py_XDECREF(torch);
    return !PyErr_Occurred();
}

}  // namespace

PyMODINIT_FUNC PyInit__native(void)
{
    if (!fits()) return nullptr;
    g_names = {PyUnicode_InternFromString("h"), PyUnicode_InternFromString("w"), PyUnicode_InternFromString("vec"),
               PyUnicode_InternFromString("_desc_ptr")};
    return PyModule_Create(&g_module);
}
