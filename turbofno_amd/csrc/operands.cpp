// Python extension `_operands`: the operand checks of the binding (turbofno_amd/api.py) and the two layer calls without a trip
// through Python per tensor attribute. A call through the ctypes binding spent 6.7 us on the host, 2.5 of them on checks and
// conversions in Python, for kernels of 5 us; through this module it spends 3.5 (S = 1, K = 8, N = 64, DY = 128, call after call:
// 6.84 -> 4.91 us).
//
// Nothing here decides that a call is wrong: whatever does not pass is handed back (None, or -1) and takes the checks in Python,
// which raise. Only plain torch.Tensor / Parameter objects are looked at, so subclasses and wrappers keep their own behaviour, and
// nothing is kept from one call to the next.
#include <torch/csrc/autograd/python_variable.h>
#include <climits>

namespace {

using Layer1d = int (*)(int, int, int, int, int, const void*, const void*, void*, float, float, void*);
using Layer2d = int (*)(int, int, int, int, int, const void*, const void*, void*, float, float, void*, size_t, int, void*);

// a contiguous tensor of that type on a GPU; the device is the one that `device` names, or becomes it if that is negative
const at::Tensor* gpu_tensor(PyObject* o, at::ScalarType type, int& device)
{
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.defined() || !t.is_cuda() || t.scalar_type() != type || !t.is_contiguous()) return nullptr;
    if (device < 0) device = t.get_device();
    return t.get_device() == device ? &t : nullptr;
}

// The interpreter's lock is given back while a launch waits for room in the queue (the caller's frame holds the operands), and taken again
// however the call ends
struct WithoutLock {
    PyThreadState* held = PyEval_SaveThread();
    ~WithoutLock() { PyEval_RestoreThread(held); }
};

bool fits_int(int64_t v) { return v >= 0 && v <= INT_MAX; }

// alpha as anything with a complex value; false leaves the question to Python
bool complex_value(PyObject* o, float& re, float& im)
{
    const Py_complex v = PyComplex_AsCComplex(o);
    if (PyErr_Occurred()) {
        PyErr_Clear();
        return false;
    }
    re = (float)v.real;
    im = (float)v.imag;
    return true;
}
bool integer_value(PyObject* o, long long& v)
{
    if (!PyLong_Check(o)) return false;
    v = PyLong_AsLongLong(o);
    if (PyErr_Occurred()) {
        PyErr_Clear();
        return false;
    }
    return true;
}
void* pointer_value(PyObject* o, bool& ok)
{
    void* p = PyLong_Check(o) ? PyLong_AsVoidPtr(o) : nullptr;
    ok = PyLong_Check(o) && !PyErr_Occurred();
    PyErr_Clear();
    return p;
}

// operands(t0, n0, t1, n1, ...): the addresses of contiguous complex64 tensors of exactly n elements each, all on one GPU, else None
PyObject* operands(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    if (count < 2 || count % 2 || count > 8) Py_RETURN_NONE;
    const void* address[4];
    int device = -1;
    try {
        for (Py_ssize_t i = 0; i < count; i += 2) {
            const at::Tensor* t = gpu_tensor(args[i], at::kComplexFloat, device);
            long long n;
            if (!t || !integer_value(args[i + 1], n) || t->numel() != n) Py_RETURN_NONE;
            address[i / 2] = t->data_ptr();
        }
    } catch (...) {
        Py_RETURN_NONE;
    }
    PyObject* tuple = PyTuple_New(count / 2);
    if (!tuple) return nullptr;
    for (Py_ssize_t i = 0; i < count / 2; ++i) PyTuple_SET_ITEM(tuple, i, PyLong_FromVoidPtr(const_cast<void*>(address[i])));
    return tuple;
}

// layer_1d(function, x, W, y, alpha, dimX, stream): the status of turbofno_layer_1d, -1 if the operands are for Python to judge
PyObject* layer_1d(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    int rc = -1;
    if (count == 7) {
        try {
            int device = -1;
            bool ok_f, ok_s;
            const auto call = reinterpret_cast<Layer1d>(pointer_value(args[0], ok_f));
            void* stream = pointer_value(args[6], ok_s);
            const at::Tensor *x = gpu_tensor(args[1], at::kComplexFloat, device), *W = gpu_tensor(args[2], at::kComplexFloat, device),
                             *y = gpu_tensor(args[3], at::kComplexFloat, device);
            float re, im;
            long long dimX;
            if (ok_f && call && ok_s && x && W && y && complex_value(args[4], re, im) && integer_value(args[5], dimX) &&
                x->dim() == 3 && W->dim() == 2 && y->dim() == 3) {
                const int64_t K = x->size(0), S = x->size(1), DY = x->size(2), N = W->size(0);
                if (W->size(1) == K && y->size(0) == N && y->size(1) == S && y->size(2) == DY && dimX > 0 && S % dimX == 0 &&
                    fits_int(K) && fits_int(S) && fits_int(DY) && fits_int(N) && fits_int(dimX)) {
                    void *px = x->data_ptr(), *pW = W->data_ptr(), *py = y->data_ptr();
                    const WithoutLock unlocked;
                    rc = call((int)(S / dimX), (int)dimX, (int)DY, (int)K, (int)N, px, pW, py, re, im, stream);
                }
            }
        } catch (...) {
            rc = -1;
        }
    }
    return PyLong_FromLong(rc);
}

// layer_2d(function, x, W, y, alpha, workspace, algo, stream): likewise for turbofno_layer_2d
PyObject* layer_2d(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    int rc = -1;
    if (count == 8) {
        try {
            int device = -1;
            bool ok_f, ok_s;
            const auto call = reinterpret_cast<Layer2d>(pointer_value(args[0], ok_f));
            void* stream = pointer_value(args[7], ok_s);
            const at::Tensor *x = gpu_tensor(args[1], at::kComplexFloat, device), *W = gpu_tensor(args[2], at::kComplexFloat, device),
                             *y = gpu_tensor(args[3], at::kComplexFloat, device), *ws = gpu_tensor(args[5], at::kByte, device);
            float re, im;
            long long algo;
            if (ok_f && call && ok_s && x && W && y && ws && complex_value(args[4], re, im) && integer_value(args[6], algo) &&
                fits_int(algo) && x->dim() == 4 && W->dim() == 2 && y->dim() == 4) {
                const int64_t K = x->size(0), bs = x->size(1), DX = x->size(2), DY = x->size(3), N = W->size(0);
                if (W->size(1) == K && y->size(0) == N && y->size(1) == bs && y->size(2) == DX && y->size(3) == DY && fits_int(K) && fits_int(bs) &&
                    fits_int(DX) && fits_int(DY) && fits_int(N)) {
                    void *px = x->data_ptr(), *pW = W->data_ptr(), *py = y->data_ptr(), *pws = ws->data_ptr();
                    const size_t bytes = (size_t)ws->numel();
                    const WithoutLock unlocked;
                    rc = call((int)bs, (int)DX, (int)DY, (int)K, (int)N, px, pW, py, re, im, pws, bytes, (int)algo, stream);
                }
            }
        } catch (...) {
            rc = -1;
        }
    }
    return PyLong_FromLong(rc);
}

PyMethodDef methods[] = {
    { "operands", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(operands)), METH_FASTCALL, "addresses of complex64 GPU tensors of given sizes, or None" },
    { "layer_1d", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(layer_1d)), METH_FASTCALL, "turbofno_layer_1d on checked tensors, or -1" },
    { "layer_2d", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(layer_2d)), METH_FASTCALL, "turbofno_layer_2d on checked tensors, or -1" },
    { nullptr, nullptr, 0, nullptr },
};
PyModuleDef module = { PyModuleDef_HEAD_INIT, "_operands", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr };

}  // namespace

// BUILT_FOR: torch and Python of the headers, "torch <version>, <SOABI>"; the binding leaves the module alone under any other
PyMODINIT_FUNC PyInit__operands(void)
{
    PyObject* m = PyModule_Create(&module);
    if (m && PyModule_AddStringConstant(m, "built_for", BUILT_FOR) < 0) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
