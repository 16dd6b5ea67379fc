// _step_table: the per-step host work of a parameter list that goes through one table of ma_tensor
// records.  Every step has to look at each parameter and its gradient (there? of the table's type?
// dense? 16-byte aligned? the same objects as in the last step?), write their addresses and ring
// positions into the records and, behind the launch, move the ring positions on.  Through the
// interpreter that was 0.32 us a tensor, more than the kernels of a small list take: 30 tensors
// 11.6 us, 148 tensors 47; here 0.04.
#include <Python.h>
#include <torch/csrc/autograd/python_variable.h>

#include <exception>

#include "../../include/microadam_hip.h"

namespace {

PyObject *key_i, *key_index;  // "I", "index"

// a tensor whose data_ptr() is where its elements lie
bool plain(const at::Tensor &t) {
    return t.defined() && !t.unsafeGetTensorImpl()->is_python_dispatch() &&
           t.layout() == at::kStrided && t.is_cuda();
}

// refresh(address, params, states, groups, dtype) -> bool
//   address  of the ma_tensor records, one per entry of params
//   params   the parameters of all groups in order, as the table was built for them
//   states   their state dictionaries
//   groups   (list of the group's parameters now, lr, weight_decay) in order
//   dtype    MA_F32 or MA_BF16
// True: p, g, index, lr and weight_decay of all records are this step's.  False, with nothing that
// matters changed, if some tensor's buffers do not admit the table this time, or if something is
// not of the usual kind; the general walk then decides, tensor by tensor.
PyObject *refresh(PyObject *, PyObject *args) {
    unsigned long long address;
    PyObject *params, *states, *groups;
    int dtype;
    if (!PyArg_ParseTuple(args, "KO!O!O!i", &address, &PyList_Type, &params, &PyList_Type, &states,
                          &PyList_Type, &groups, &dtype))
        return nullptr;
    ma_tensor *rec = reinterpret_cast<ma_tensor *>(static_cast<uintptr_t>(address));
    const Py_ssize_t n = PyList_GET_SIZE(params);
    if (PyList_GET_SIZE(states) != n) Py_RETURN_FALSE;
    const at::ScalarType type = dtype == MA_BF16 ? at::kBFloat16 : at::kFloat;
    try {
        Py_ssize_t i = 0;
        for (Py_ssize_t gi = 0; gi < PyList_GET_SIZE(groups); ++gi) {
            PyObject *group = PyList_GET_ITEM(groups, gi);
            if (!PyTuple_Check(group) || PyTuple_GET_SIZE(group) != 3) Py_RETURN_FALSE;
            PyObject *list = PyTuple_GET_ITEM(group, 0);
            PyObject *lr = PyTuple_GET_ITEM(group, 1), *wd = PyTuple_GET_ITEM(group, 2);
            if (!PyList_Check(list) || !(PyFloat_Check(lr) || PyLong_Check(lr)) ||
                !(PyFloat_Check(wd) || PyLong_Check(wd)))
                Py_RETURN_FALSE;
            const double lr_value = PyFloat_AsDouble(lr), wd_value = PyFloat_AsDouble(wd);
            if (PyErr_Occurred()) return nullptr;
            for (Py_ssize_t j = 0; j < PyList_GET_SIZE(list); ++j, ++i) {
                if (i >= n || PyList_GET_ITEM(list, j) != PyList_GET_ITEM(params, i))
                    Py_RETURN_FALSE;
                PyObject *obj = PyList_GET_ITEM(params, i), *st = PyList_GET_ITEM(states, i);
                if (!THPVariable_Check(obj) || !PyDict_Check(st)) Py_RETURN_FALSE;
                const at::Tensor &p = THPVariable_Unpack(obj);
                if (!plain(p)) Py_RETURN_FALSE;
                const at::Tensor &g = p.grad();
                if (!plain(g) || p.scalar_type() != type || g.scalar_type() != type ||
                    !p.is_contiguous() || !g.is_contiguous())
                    Py_RETURN_FALSE;
                PyObject *window = PyDict_GetItemWithError(st, key_i);
                PyObject *index = PyDict_GetItemWithError(st, key_index);
                if (!window || !index) {
                    if (PyErr_Occurred()) return nullptr;
                    Py_RETURN_FALSE;
                }
                if (!THPVariable_Check(window) || !PyLong_Check(index) ||
                    THPVariable_Unpack(window).scalar_type() != at::kShort)
                    Py_RETURN_FALSE;
                const long row = PyLong_AsLong(index);
                if (row == -1 && PyErr_Occurred()) return nullptr;
                if (row != static_cast<int32_t>(row)) Py_RETURN_FALSE;  // (refused by the walk)
                void *pp = p.data_ptr(), *gp = g.data_ptr();
                if (((reinterpret_cast<uintptr_t>(pp) | reinterpret_cast<uintptr_t>(gp)) & 15) != 0)
                    Py_RETURN_FALSE;
                rec[i].p = pp;
                rec[i].g = gp;
                rec[i].index = static_cast<int32_t>(row);
                rec[i].lr = lr_value;
                rec[i].weight_decay = wd_value;
            }
        }
        if (i != n) Py_RETURN_FALSE;
    } catch (const std::exception &e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
        return nullptr;
    }
    Py_RETURN_TRUE;
}

// (value + 1) % m as the interpreter forms it, for ring positions that are not plain integers
PyObject *advanced(PyObject *value, long m) {
    Py_INCREF(value);
    PyObject *one = PyLong_FromLong(1), *length = PyLong_FromLong(m);
    PyObject *sum = one && length ? PyNumber_Add(value, one) : nullptr;
    PyObject *next = sum ? PyNumber_Remainder(sum, length) : nullptr;
    Py_XDECREF(one);
    Py_XDECREF(length);
    Py_XDECREF(sum);
    Py_DECREF(value);
    return next;
}

// advance(states, m): state['index'] = (state['index'] + 1) % m (micro_adam.py:211), whatever kind of
// number the position is: the step has been launched, and what it took must not fail here (a
// framework that re-types optimizer state may have made a float or a tensor of it).
PyObject *advance(PyObject *, PyObject *args) {
    PyObject *states;
    long m;
    if (!PyArg_ParseTuple(args, "O!l", &PyList_Type, &states, &m)) return nullptr;
    if (m < 1) {
        PyErr_SetString(PyExc_ValueError, "a window has at least one row");
        return nullptr;
    }
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(states); ++i) {
        PyObject *st = PyList_GET_ITEM(states, i);
        PyObject *index = PyDict_Check(st) ? PyDict_GetItemWithError(st, key_index) : nullptr;
        if (!index) {
            if (!PyErr_Occurred()) PyErr_SetString(PyExc_KeyError, "index");
            return nullptr;
        }
        const long row = PyLong_CheckExact(index) ? PyLong_AsLong(index) : -1;
        if (row == -1) PyErr_Clear();
        PyObject *next =
            row >= 0 && row < m ? PyLong_FromLong((row + 1) % m) : advanced(index, m);
        if (!next) return nullptr;
        const int rc = PyDict_SetItem(st, key_index, next);
        Py_DECREF(next);
        if (rc) return nullptr;
    }
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"refresh", refresh, METH_VARARGS, "this step's buffers and hyper-parameters into the records"},
    {"advance", advance, METH_VARARGS, "the ring positions behind a step"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_step_table", nullptr, -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__step_table(void) {
    key_i = PyUnicode_InternFromString("I");
    key_index = PyUnicode_InternFromString("index");
    if (!key_i || !key_index) return nullptr;
    return PyModule_Create(&module);
}
