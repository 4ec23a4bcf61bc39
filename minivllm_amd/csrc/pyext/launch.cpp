// Calls of C functions by address from Python, for the launchers of the kernel libraries: `bind(address, types)` is a
// callable that turns its arguments into machine words and makes the call with the interpreter's lock released.  ctypes does
// the same with an object and a conversion table for every argument: a launcher of 25 arguments costs 4.6 us a call
// through it and 0.4 like this, where the smallest attention call takes 10 to 13 us altogether.
//
// `types`: a letter per argument, p - a pointer (an int, or None for 0), i - an integer (of either sign, taken modulo 2^64),
// f - a float; then one for the result, I (int) or L (long).  What is none of it is a TypeError, as through ctypes.  x86-64 System V only: there integers go to six
// registers and then to the stack in their order, floats to registers of their own (up to eight here), so that every
// signature is called through one type; words on the stack that a function does not have are the caller's to remove.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stdint.h>

#if !defined(__x86_64__) || defined(_WIN32)
#error "the calling convention below is that of x86-64 System V"
#endif

namespace {

constexpr int REGS = 6, STACK = 40, FLOATS = 8, ARGS = 48;

struct Call {
    void* fn;
    int n;
    bool wide;                  // the result is a long
    char types[ARGS];
};

typedef long (*Any)(uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, float, float, float, float, float, float,
                    float, float, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t,
                    uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t,
                    uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t,
                    uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t,
                    uint64_t);

PyObject* call(PyObject* self, PyObject* const* args, Py_ssize_t n) {
    const Call* c = static_cast<const Call*>(PyCapsule_GetPointer(self, nullptr));
    if (!c) return nullptr;
    if (n != c->n) {
        PyErr_Format(PyExc_TypeError, "%d arguments expected, got %zd", c->n, n);
        return nullptr;
    }
    uint64_t w[REGS + STACK] = {0};
    float f[FLOATS] = {0};
    int nw = 0, nf = 0;
    for (Py_ssize_t i = 0; i < n; ++i) {
        if (c->types[i] == 'f') {
            const double x = PyFloat_AsDouble(args[i]);
            if (x == -1.0 && PyErr_Occurred()) return nullptr;
            f[nf++] = (float)x;
        } else if (c->types[i] == 'p' && args[i] == Py_None) {
            w[nw++] = 0;
        } else {
            if (c->types[i] == 'p' && !PyLong_Check(args[i])) {
                PyErr_Format(PyExc_TypeError, "argument %zd: a pointer expected, an int or None", i + 1);
                return nullptr;
            }
            if (PyFloat_Check(args[i])) {
                PyErr_Format(PyExc_TypeError, "argument %zd: int expected instead of float", i + 1);
                return nullptr;
            }
            const uint64_t x = PyLong_AsUnsignedLongLongMask(args[i]);
            if (x == (uint64_t)-1 && PyErr_Occurred()) return nullptr;
            w[nw++] = x;
        }
    }
    long r;
    Py_BEGIN_ALLOW_THREADS
    const uint64_t* s = w + REGS;
    r = reinterpret_cast<Any>(c->fn)(
        w[0], w[1], w[2], w[3], w[4], w[5], f[0], f[1], f[2], f[3], f[4], f[5], f[6], f[7], s[0], s[1], s[2], s[3], s[4],
        s[5], s[6], s[7], s[8], s[9], s[10], s[11], s[12], s[13], s[14], s[15], s[16], s[17], s[18], s[19], s[20], s[21],
        s[22], s[23], s[24], s[25], s[26], s[27], s[28], s[29], s[30], s[31], s[32], s[33], s[34], s[35], s[36], s[37],
        s[38], s[39]);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(c->wide ? r : (long)(int)r);
}

PyMethodDef call_def = {"launcher", (PyCFunction)(void (*)(void))call, METH_FASTCALL, nullptr};

void drop(PyObject* capsule) { PyMem_Free(PyCapsule_GetPointer(capsule, nullptr)); }

PyObject* bind(PyObject*, PyObject* args) {
    unsigned long long address;
    const char* types;
    Py_ssize_t len;
    if (!PyArg_ParseTuple(args, "Ks#", &address, &types, &len)) return nullptr;
    int words = 0, floats = 0;
    bool ok = address != 0 && len >= 1 && len - 1 <= ARGS && (types[len - 1] == 'I' || types[len - 1] == 'L');
    for (Py_ssize_t i = 0; ok && i + 1 < len; ++i) {
        floats += types[i] == 'f';
        words += types[i] != 'f';
        ok = types[i] == 'p' || types[i] == 'i' || types[i] == 'f';
    }
    if (!ok || words > REGS + STACK || floats > FLOATS) {
        PyErr_SetString(PyExc_ValueError, "no such call");
        return nullptr;
    }
    Call* c = static_cast<Call*>(PyMem_Calloc(1, sizeof(Call)));
    if (!c) return PyErr_NoMemory();
    c->fn = reinterpret_cast<void*>(address);
    c->n = (int)len - 1;
    c->wide = types[len - 1] == 'L';
    for (int i = 0; i < c->n; ++i) c->types[i] = types[i];
    PyObject* self = PyCapsule_New(c, nullptr, drop);
    if (!self) {
        PyMem_Free(c);
        return nullptr;
    }
    PyObject* f = PyCFunction_New(&call_def, self);
    Py_DECREF(self);
    return f;
}

PyMethodDef methods[] = {{"bind", bind, METH_VARARGS, "bind(address, types) -> callable"}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_launch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__launch(void) { return PyModule_Create(&module); }
