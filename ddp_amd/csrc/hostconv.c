/* Conversion of update lines from Python objects to the ABI's structs.
 *
 * A batch of 20,000 (flag, u, v, w) tuples took 5 to 10 ms to convert with one
 * ctypes attribute store per field, ten times what applying it takes; reading
 * the objects through the C API takes 0.5 ms. */
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stdint.h>

/* fill(lines, out): writes lines[i][0..3] into the writable buffer out as four
 * 32-bit words each, reduced modulo 2^32 as a ctypes store does.  Takes lists
 * and tuples of lists and tuples of ints; returns False on anything else, with
 * the caller to convert it by the general rules. */
static PyObject *fill(PyObject *self, PyObject *args)
{
    PyObject *lines;
    Py_buffer out;
    if (!PyArg_ParseTuple(args, "Ow*", &lines, &out)) return NULL;
    int ok = PyList_CheckExact(lines) || PyTuple_CheckExact(lines);
    const Py_ssize_t n = ok ? PySequence_Fast_GET_SIZE(lines) : 0;
    if (n > out.len / 16) ok = 0;
    uint32_t *dst = (uint32_t *)out.buf;
    for (Py_ssize_t i = 0; ok && i < n; ++i) {
        PyObject *l = PySequence_Fast_GET_ITEM(lines, i);
        if (!(PyTuple_CheckExact(l) || PyList_CheckExact(l)) || PySequence_Fast_GET_SIZE(l) < 4) {
            ok = 0;
            break;
        }
        for (int k = 0; k < 4; ++k) {
            PyObject *x = PySequence_Fast_GET_ITEM(l, k);
            int overflow = 0;
            if (!PyLong_CheckExact(x)) {
                ok = 0;
                break;
            }
            const long long v = PyLong_AsLongLongAndOverflow(x, &overflow);
            if (overflow) {
                ok = 0;
                break;
            }
            dst[4 * i + k] = (uint32_t)(uint64_t)v;
        }
    }
    PyBuffer_Release(&out);
    return PyBool_FromLong(ok);
}

static PyMethodDef methods[] = {{"fill", fill, METH_VARARGS, "fill(lines, out) -> bool"}, {NULL, NULL, 0, NULL}};
static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_hostconv", NULL, -1, methods, NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit__hostconv(void) { return PyModule_Create(&module); }
