/* The per-token calls of include/saragossa_kv.h as Python functions.
 *
 * A decode step is two launches of a few microseconds; ctypes took 1.6 us for the fifteen arguments of
 * one (0.25 us here), three calls per layer in a chunk. Each function takes the C call's arguments:
 * pointers, handles and sizes as int (or None for a null pointer) and floats as float, releases the
 * interpreter lock around the call as ctypes does, and returns its status code; -1, without calling
 * anything, where an argument is of another type: the caller then goes through ctypes, which takes or
 * refuses what it always has.
 */
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include "../../include/saragossa_kv.h"

/* an int as ctypes reads it into a pointer or a size (modulo 2^64) */
static int word(PyObject *o, uint64_t *out) {
    if (!PyLong_CheckExact(o)) return 0;
    *out = PyLong_AsUnsignedLongLongMask(o);
    return 1;
}

/* Arguments by kind: p = pointer or None, n = size, f = float; words and floats in the order they stand. */
static int take(PyObject *const *args, Py_ssize_t n, const char *kinds, uint64_t *w, float *f) {
    Py_ssize_t i;
    for (i = 0; kinds[i]; ++i) {
        if (i >= n) return 0;
        if (kinds[i] == 'f') {
            if (!PyFloat_CheckExact(args[i])) return 0;
            *f++ = (float)PyFloat_AS_DOUBLE(args[i]);
        } else {
            if (kinds[i] == 'p' && args[i] == Py_None) *w = 0;
            else if (!word(args[i], w)) return 0;
            ++w;
        }
    }
    return i == n;
}

#define P(i) ((void *)(uintptr_t)w[i])
#define N(i) ((size_t)w[i])
#define CALL(name, kinds, expr)                                                            \
    static PyObject *name(PyObject *self, PyObject *const *args, Py_ssize_t nargs) {       \
        uint64_t w[16];                                                                    \
        float f[2];                                                                        \
        int32_t rc;                                                                        \
        (void)self;                                                                        \
        (void)f;                                                                           \
        if (!take(args, nargs, kinds, w, f)) return PyLong_FromLong(-1);                   \
        Py_BEGIN_ALLOW_THREADS                                                             \
        rc = (expr);                                                                       \
        Py_END_ALLOW_THREADS                                                               \
        return PyLong_FromLong(rc);                                                        \
    }

CALL(truncate_rows, "pn", skv_truncate(P(0), N(1)))
CALL(append_batch, "ppppn", skv_append_batch_device(P(0), P(1), P(2), P(3), N(4)))
CALL(attention, "ppppn", skv_attention_device(P(0), P(1), P(2), P(3), N(4)))
CALL(decode_step, "pppnpnpp", skv_decode_step_device(P(0), P(1), P(2), N(3), P(4), N(5), P(6), P(7)))
CALL(decode_step_prekv, "pppnpnpnpnppffp",
     skv_decode_step_prekv_device(P(0), P(1), P(2), N(3), P(4), N(5), P(6), N(7), P(8), N(9), P(10), P(11), f[0], f[1], P(12)))
CALL(decode_step_gated, "pppnpnpnpnppffp",
     skv_decode_step_gated_device(P(0), P(1), P(2), N(3), P(4), N(5), P(6), N(7), P(8), N(9), P(10), P(11), f[0], f[1], P(12)))
CALL(prefill_chunk, "pppppnp", skv_prefill_chunk_device(P(0), P(1), P(2), P(3), P(4), N(5), P(6)))
CALL(rms_norm_rope_rows, "pppnppnnnfp",
     skv_rms_norm_rope_rows_device(P(0), P(1), P(2), N(3), P(4), P(5), N(6), N(7), N(8), f[0], P(9)))

#define ENTRY(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, NULL}
static PyMethodDef methods[] = {ENTRY(truncate_rows),     ENTRY(append_batch),      ENTRY(attention),
                                ENTRY(decode_step),       ENTRY(decode_step_prekv), ENTRY(decode_step_gated),
                                ENTRY(prefill_chunk),     ENTRY(rms_norm_rope_rows), {NULL, NULL, 0, NULL}};

static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_calls", NULL, 0, methods, NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit__calls(void) { return PyModule_Create(&module); }
