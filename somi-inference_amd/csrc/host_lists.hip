// Python lists of token ids as one array, for the copy to the device: an element costs 3 ns here and 20 to 50 through array, numpy
// or torch constructors (64 histories of 700 ids: 45,000 elements a sampled step).  Host code only.
//
// The interpreter's functions come from the process that loaded the library (names and signatures of the stable C API); the
// caller holds the interpreter's lock (ctypes.PyDLL).
#include "common.h"

extern "C" {
typedef struct _object PyObject;
__attribute__((weak)) intptr_t PyList_Size(PyObject*);
__attribute__((weak)) PyObject* PyList_GetItem(PyObject*, intptr_t);       // borrowed
__attribute__((weak)) long PyLong_AsLong(PyObject*);
__attribute__((weak)) PyObject* PyErr_Occurred(void);
}

// lists: a list of lists of integers; out: their elements one after another, `capacity` of them at most.  Returns how many there are,
// -1 with a Python exception set, -2 where an element does not fit 32 bits, -3 where there is no room or no interpreter.
extern "C" int64_t somi_gather_ids(PyObject* lists, int32_t* out, int64_t capacity) {
    if (!PyList_Size || !PyList_GetItem || !PyLong_AsLong || !PyErr_Occurred) return -3;
    const intptr_t rows = PyList_Size(lists);
    if (rows < 0) return -1;
    int64_t at = 0;
    for (intptr_t row = 0; row < rows; ++row) {
        PyObject* list = PyList_GetItem(lists, row);
        if (list == nullptr) return -1;
        const intptr_t count = PyList_Size(list);
        if (count < 0) return -1;
        if (at + count > capacity) return -3;
        for (intptr_t i = 0; i < count; ++i) {
            PyObject* item = PyList_GetItem(list, i);      // (a list that an element's own code shortens ends here)
            if (item == nullptr) return -1;
            const long value = PyLong_AsLong(item);
            if (value == -1 && PyErr_Occurred()) return -1;
            if (value < INT32_MIN || value > INT32_MAX) return -2;
            out[at++] = (int32_t)value;
        }
    }
    return at;
}
