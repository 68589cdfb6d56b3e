// A step's inputs out of its batch entries: the tokens, counts, slots and wanted places of a plain batch read from the Python
// objects in one pass; step_rows.cpp lays them out for the device.  All of it is before the GPU has anything to do: entry by entry in
// Python a step of 64 single tokens took 53 us for the first and 19 for the second, 198 from its call to the captured graph's launch;
// here 5 and 2, and with the block tables' rows in one copy (../upload.hip) 48.
//
// Called through ctypes.PyDLL, so with the interpreter's lock held.  Raises nothing: what is not a plain batch is left to the
// caller, which refuses it with the precise error or takes its odd forms; it also takes every batch where this file could not be
// compiled for want of the interpreter's headers.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstdint>

namespace {

// The elements of a list or tuple (borrowed; an empty list has no array of them); false for anything else.
bool items(PyObject* o, PyObject*** v, Py_ssize_t* n) {
    if (PyList_CheckExact(o)) {
        *n = PyList_GET_SIZE(o);
        *v = reinterpret_cast<PyListObject*>(o)->ob_item;
        return true;
    }
    if (PyTuple_CheckExact(o)) {
        *n = PyTuple_GET_SIZE(o);
        *v = reinterpret_cast<PyTupleObject*>(o)->ob_item;
        return true;
    }
    return false;
}

// A whole number in [0, limit), or -1.
long whole(PyObject* o, long limit) {
    if (!PyLong_CheckExact(o)) return -1;
    int overflow = 0;
    const long v = PyLong_AsLongAndOverflow(o, &overflow);
    return overflow == 0 && v >= 0 && v < limit ? v : -1;
}

struct Ref {                                  // a new reference, given back
    PyObject* o;
    explicit Ref(PyObject* p) : o(p) {}
    ~Ref() { Py_XDECREF(o); }
    Ref(const Ref&) = delete;
};

}  // namespace

extern "C" {

// entries: a list of objects with `slot`, `tokens` and `want`.  Writes the tokens one entry behind the other (room for max_tokens),
// per entry its number of tokens, slot and number of wanted places (room for max_tokens each), and the wanted rows of the batch (room
// for max_rows); totals: entries, tokens, wanted rows, and whether every entry is one token that wants its logits.
// 0: done.  1: not a plain batch (lists or tuples of whole numbers inside their bounds, places ascending, within the limits).
int mlr_step_entries(PyObject* entries, long vocab, int max_tokens, int max_rows, int32_t* ids, int32_t* counts, int32_t* slots,
                     int32_t* want_counts, int32_t* want_rows, int32_t* totals) {
    static PyObject* const slot_name = PyUnicode_InternFromString("slot");
    static PyObject* const tokens_name = PyUnicode_InternFromString("tokens");
    static PyObject* const want_name = PyUnicode_InternFromString("want");
    if (slot_name == nullptr || tokens_name == nullptr || want_name == nullptr) {
        PyErr_Clear();
        return 1;
    }
    if (!PyList_CheckExact(entries)) return 1;
    int total = 0, rows = 0, n = 0;
    bool single = true;
    for (; n < PyList_GET_SIZE(entries); ++n) {              // (an attribute may be code that changes the list)
        PyObject* e = PyList_GET_ITEM(entries, n);
        Py_INCREF(e);
        const Ref entry(e), slot(PyObject_GetAttr(e, slot_name)), tokens(PyObject_GetAttr(e, tokens_name)), want(PyObject_GetAttr(e, want_name));
        if (slot.o == nullptr || tokens.o == nullptr || want.o == nullptr) {
            PyErr_Clear();
            return 1;
        }
        Py_ssize_t n_tokens = 0, n_want = 0;
        PyObject **t = nullptr, **w = nullptr;
        if (!items(tokens.o, &t, &n_tokens) || !items(want.o, &w, &n_want)) return 1;
        const long s = whole(slot.o, 0x7fffffffL);
        if (s < 0 || n_tokens < 1 || n_tokens > max_tokens - total || n_want > max_rows - rows) return 1;
        for (Py_ssize_t i = 0; i < n_tokens; ++i) {
            const long v = whole(t[i], vocab);
            if (v < 0) return 1;
            ids[total + i] = (int32_t)v;
        }
        long before = -1;
        for (Py_ssize_t i = 0; i < n_want; ++i) {
            const long v = whole(w[i], (long)n_tokens);
            if (v <= before) return 1;
            want_rows[rows + i] = (int32_t)(total + v);
            before = v;
        }
        single = single && n_tokens == 1 && n_want == 1;
        counts[n] = (int32_t)n_tokens;
        slots[n] = (int32_t)s;
        want_counts[n] = (int32_t)n_want;
        total += (int)n_tokens;
        rows += (int)n_want;
    }
    if (n == 0) return 1;
    totals[0] = n;
    totals[1] = total;
    totals[2] = rows;
    totals[3] = single ? 1 : 0;
    return 0;
}

}  // extern "C"
