/* CPython entry to the functions of librocwmma_amd.so that a program calls over and over.
 *
 * Each function takes the arguments of the C function it is named after, device pointers as tensors (anything with data_ptr()),
 * plain addresses or None, and returns its status.  ctypes converts twenty arguments through as many objects: a call of
 * rocwmma_amd.gemm took 4.8 us of host time, 2.4 of them in ctypes and 0.8 in its preparation, more than the kernel of a 256^3 product
 * takes on the device.  bind() is given the address of a C function and its ctypes object, which gets whatever is not a plain
 * Python number (it converts or refuses it as ever).  As with ctypes, other threads run during a call.
 *
 * rocwmma_amd.gemm with a function that does nothing 4.8 -> 1.0 us; 256^3 f16 with C, launches one behind the other, 6.2 -> 4.9. */
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stdint.h>

#define MAX_ARGS 24

enum
{
    GEMM_EX,
    GEMM_BIAS_ACT,
    GEMM_MX,
    GEMV,
    DLRM_FWD_EX,
    DLRM_BWD_EX,
    FUNCTIONS
};

/* i: int or uint32_t (masked as ctypes does), p: pointer, z: size_t, f: float */
static const struct
{
    const char* name;
    const char* args;
} kFunctions[FUNCTIONS] = {{"gemm_ex", "iiiiiiiiipipipipiffp"}, {"gemm_bias_act", "iiiiiiiipipipipiffpip"}, {"gemm_mx", "iiiiiiipipipipipipiffpzp"},
                           {"gemv", "iiipipipiffp"},            {"dlrm_fwd_ex", "ippiiip"},                  {"dlrm_bwd_ex", "ippppiiip"}};

static void*     address[FUNCTIONS];
static PyObject* slow[FUNCTIONS]; /* the ctypes function */
static PyObject* dataPtr; /* "data_ptr" */

/* The general way: the ctypes function on the same arguments, pointers taken out of their tensors. */
static PyObject* callSlow(int which, PyObject* const* args, Py_ssize_t count)
{
    const char*      form      = kFunctions[which].args;
    const Py_ssize_t known     = (Py_ssize_t)strlen(form);
    PyObject*        converted = PyTuple_New(count);
    PyObject*        result;
    Py_ssize_t       i;
    if(!converted)
        return NULL;
    for(i = 0; i < count; ++i)
    {
        PyObject* v = args[i];
        if(i < known && form[i] == 'p' && v != Py_None && !PyLong_Check(v) && PyObject_HasAttr(v, dataPtr))
        {
            v = PyObject_CallMethodNoArgs(v, dataPtr);
            if(!v)
            {
                Py_DECREF(converted);
                return NULL;
            }
        }
        else
            Py_INCREF(v);
        PyTuple_SET_ITEM(converted, i, v);
    }
    result = PyObject_CallObject(slow[which], converted);
    Py_DECREF(converted);
    return result;
}

/* 1: converted, 0: something that ctypes has to look at, -1: an error is set */
static int convert(const char* form, PyObject* const* args, Py_ssize_t count, uint64_t* word, float* real)
{
    Py_ssize_t i;
    int        reals = 0;
    for(i = 0; i < count; ++i)
    {
        PyObject* v = args[i];
        if(form[i] == 'f')
        {
            if(!PyFloat_CheckExact(v))
                return 0;
            real[reals++] = (float)PyFloat_AS_DOUBLE(v);
        }
        else if(PyLong_CheckExact(v))
            word[i] = PyLong_AsUnsignedLongLongMask(v);
        else if(form[i] != 'p')
            return 0;
        else if(v == Py_None)
            word[i] = 0;
        else
        {
            PyObject* at = PyObject_CallMethodNoArgs(v, dataPtr);
            if(!at)
            {
                if(!PyErr_ExceptionMatches(PyExc_AttributeError))
                    return -1;
                PyErr_Clear();
                return 0;
            }
            if(!PyLong_CheckExact(at))
            {
                Py_DECREF(at);
                return 0;
            }
            word[i] = PyLong_AsUnsignedLongLongMask(at);
            Py_DECREF(at);
        }
    }
    return 1;
}

#define I(n) ((int)w[n])
#define U(n) ((uint32_t)w[n])
#define P(n) ((void*)(uintptr_t)w[n])
typedef uint32_t u32;

static int run(int which, const uint64_t* w, const float* f)
{
    void* at = address[which];
    switch(which)
    {
    case GEMM_EX:
        return ((int (*)(int, int, int, int, int, int, u32, u32, u32, void*, u32, void*, u32, void*, u32, void*, u32, float, float, void*))at)(
            I(0), I(1), I(2), I(3), I(4), I(5), U(6), U(7), U(8), P(9), U(10), P(11), U(12), P(13), U(14), P(15), U(16), f[0], f[1], P(19));
    case GEMM_BIAS_ACT:
        return ((int (*)(int, int, int, int, int, u32, u32, u32, void*, u32, void*, u32, void*, u32, void*, u32, float, float, void*, int, void*))at)(
            I(0), I(1), I(2), I(3), I(4), U(5), U(6), U(7), P(8), U(9), P(10), U(11), P(12), U(13), P(14), U(15), f[0], f[1], P(18), I(19), P(20));
    case GEMM_MX:
        return ((int (*)(int, int, int, int, u32, u32, u32, void*, u32, void*, u32, void*, u32, void*, u32, void*, u32, void*, u32, float, float, void*,
                         size_t, void*))at)(I(0), I(1), I(2), I(3), U(4), U(5), U(6), P(7), U(8), P(9), U(10), P(11), U(12), P(13), U(14), P(15), U(16),
                                            P(17), U(18), f[0], f[1], P(21), (size_t)w[22], P(23));
    case GEMV:
        return ((int (*)(u32, u32, u32, void*, u32, void*, u32, void*, u32, float, float, void*))at)(U(0), U(1), U(2), P(3), U(4), P(5), U(6), P(7), U(8),
                                                                                                    f[0], f[1], P(11));
    case DLRM_FWD_EX:
        return ((int (*)(int, void*, void*, u32, u32, u32, void*))at)(I(0), P(1), P(2), U(3), U(4), U(5), P(6));
    default:
        return ((int (*)(int, void*, void*, void*, void*, u32, u32, u32, void*))at)(I(0), P(1), P(2), P(3), P(4), U(5), U(6), U(7), P(8));
    }
}

static PyObject* call(int which, PyObject* const* args, Py_ssize_t count)
{
    uint64_t word[MAX_ARGS] = {0};
    float    real[2]        = {0.0f, 0.0f};
    int      rc;
    if(!address[which])
    {
        PyErr_SetString(PyExc_RuntimeError, "not bound to the library");
        return NULL;
    }
    if((size_t)count != strlen(kFunctions[which].args))
        return callSlow(which, args, count);
    rc = convert(kFunctions[which].args, args, count, word, real);
    if(rc < 0)
        return NULL;
    if(rc == 0)
        return callSlow(which, args, count);
    Py_BEGIN_ALLOW_THREADS
    rc = run(which, word, real);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
}

#define ENTRY(name, which)                                                            \
    static PyObject* name(PyObject* self, PyObject* const* args, Py_ssize_t count)    \
    {                                                                                 \
        (void)self;                                                                   \
        return call(which, args, count);                                              \
    }
ENTRY(gemmEx, GEMM_EX)
ENTRY(gemmBiasAct, GEMM_BIAS_ACT)
ENTRY(gemmMx, GEMM_MX)
ENTRY(gemvCall, GEMV)
ENTRY(dlrmFwdEx, DLRM_FWD_EX)
ENTRY(dlrmBwdEx, DLRM_BWD_EX)

/* bind(name, address, ctypes function) */
static PyObject* bindFunction(PyObject* self, PyObject* args)
{
    const char*        name;
    unsigned long long at;
    PyObject*          function;
    int                which;
    (void)self;
    if(!PyArg_ParseTuple(args, "sKO", &name, &at, &function))
        return NULL;
    for(which = 0; which < FUNCTIONS; ++which)
        if(strcmp(name, kFunctions[which].name) == 0)
        {
            Py_INCREF(function);
            Py_XSETREF(slow[which], function);
            address[which] = (void*)(uintptr_t)at;
            Py_RETURN_NONE;
        }
    PyErr_Format(PyExc_KeyError, "%s", name);
    return NULL;
}

static PyMethodDef methods[] = {{"bind", bindFunction, METH_VARARGS, "bind(name, address, ctypes function)"},
                                {"gemm_ex", (PyCFunction)(void*)gemmEx, METH_FASTCALL, "rocwmma_amd_gemm_ex"},
                                {"gemm_bias_act", (PyCFunction)(void*)gemmBiasAct, METH_FASTCALL, "rocwmma_amd_gemm_bias_act"},
                                {"gemm_mx", (PyCFunction)(void*)gemmMx, METH_FASTCALL, "rocwmma_amd_gemm_mx"},
                                {"gemv", (PyCFunction)(void*)gemvCall, METH_FASTCALL, "rocwmma_amd_gemv"},
                                {"dlrm_fwd_ex", (PyCFunction)(void*)dlrmFwdEx, METH_FASTCALL, "rocwmma_amd_dlrm_fwd_ex"},
                                {"dlrm_bwd_ex", (PyCFunction)(void*)dlrmBwdEx, METH_FASTCALL, "rocwmma_amd_dlrm_bwd_ex"},
                                {NULL, NULL, 0, NULL}};

static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_calls", "The library's functions without ctypes", -1, methods, NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit__calls(void)
{
    dataPtr = PyUnicode_InternFromString("data_ptr");
    return dataPtr ? PyModule_Create(&module) : NULL;
}
