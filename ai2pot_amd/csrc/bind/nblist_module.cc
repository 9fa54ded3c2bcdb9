// CPython extension module `nblist` with the reference module's single function
//   find_info4mlff(lattice, types, coords, rcut, umax, is_cart, pbc_xyz, sort)
//       -> (inum, ilist, numneigh, firstneigh, rcs, types, nghost)
// (source/nblist/bind/nblist_bind.cc:35-207): same positional signature, same type checks
// (TypeError), NumPy arrays in and out, float32 / float64 selected by the dtype of coords.
// The list is built on the current HIP device by libai2pot_hip.so (a2p_nblist_host_into_*); the arrays
// returned are ordinary NumPy arrays.  Unlike the reference, more than `umax` neighbours raises
// RuntimeError instead of overrunning the output arrays.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#define NPY_NO_DEPRECATED_API NPY_1_7_API_VERSION
#include <numpy/arrayobject.h>
#include <string>

#include "../../../include/ai2pot_hip.h"

namespace {

PyObject* fail(PyObject* exc, const std::string& msg)
{
    PyErr_SetString(exc, msg.c_str());
    return nullptr;
}

PyObject* run(PyArrayObject* lattice, PyArrayObject* types, PyArrayObject* coords, double rcut, int umax,
              bool is_cart, const int* pbc, bool sort, int npy_float)
{
    const int n = (int)PyArray_DIM(coords, 0);
    if (n <= 0) return fail(PyExc_RuntimeError, "the structure has no atoms");
    npy_intp d1[1] = {n}, d2[2] = {n, umax}, d3[3] = {n, umax, 3};
    PyObject* ilist = PyArray_SimpleNew(1, d1, NPY_INT32);
    PyObject* nn = PyArray_SimpleNew(1, d1, NPY_INT32);
    PyObject* first = PyArray_SimpleNew(2, d2, NPY_INT32);
    PyObject* rcs = PyArray_SimpleNew(3, d3, npy_float);
    PyObject* tout = PyArray_SimpleNew(1, d1, NPY_INT32);
    auto drop = [&]() -> PyObject* {
        Py_XDECREF(ilist); Py_XDECREF(nn); Py_XDECREF(first); Py_XDECREF(rcs); Py_XDECREF(tout);
        return nullptr;
    };
    if (!(ilist && nn && first && rcs && tout)) return drop();
    auto data = [](PyObject* a) { return PyArray_DATA((PyArrayObject*)a); };
    int most = 0;
    const int rc = npy_float == NPY_FLOAT32
        ? a2p_nblist_host_into_f32((const float*)PyArray_DATA(lattice), (const int*)PyArray_DATA(types),
                                   (const float*)PyArray_DATA(coords), n, rcut, umax, is_cart, pbc, sort, (int*)data(ilist),
                                   (int*)data(nn), (int*)data(first), (float*)data(rcs), (int*)data(tout), &most)
        : a2p_nblist_host_into_f64((const double*)PyArray_DATA(lattice), (const int*)PyArray_DATA(types),
                                   (const double*)PyArray_DATA(coords), n, rcut, umax, is_cart, pbc, sort, (int*)data(ilist),
                                   (int*)data(nn), (int*)data(first), (double*)data(rcs), (int*)data(tout), &most);
    if (rc != A2P_OK) {
        drop();
        return fail(PyExc_RuntimeError, std::string("libai2pot_hip: ") + a2p_last_error());
    }
    return Py_BuildValue("(iNNNNNi)", n, ilist, nn, first, rcs, tout, 0);
}

PyObject* py_find_info4mlff(PyObject*, PyObject* args)
{
    PyObject *lat, *types_in, *coords, *rcut, *umax, *is_cart, *pbc, *sort;
    if (!PyArg_ParseTuple(args, "OOOOOOOO", &lat, &types_in, &coords, &rcut, &umax, &is_cart, &pbc, &sort))
        return nullptr;
    if (!PyArray_Check(lat) || !PyArray_Check(types_in) || !PyArray_Check(coords) || !PyFloat_Check(rcut) ||
        !PyLong_Check(umax) || PyBool_Check(umax) || !PyBool_Check(is_cart) || !PyList_Check(pbc) ||
        !PyBool_Check(sort))
        return fail(PyExc_TypeError, "Please check the parameter in interface of py_find_info4mlff().");
    if (PyList_Size(pbc) != 3) return fail(PyExc_TypeError, "pbc_xyz must have three entries");
    const int ft = PyArray_TYPE((PyArrayObject*)coords);
    if ((ft != NPY_FLOAT32 && ft != NPY_FLOAT64) || PyArray_TYPE((PyArrayObject*)lat) != ft)
        return fail(PyExc_TypeError, "lattice and coords must share dtype float32 or float64");
    const int it = PyArray_TYPE((PyArrayObject*)types_in);
    if (it != NPY_INT32 && it != NPY_INT64) return fail(PyExc_TypeError, "types must be int32 or int64");
    if (PyArray_NDIM((PyArrayObject*)coords) != 2 || PyArray_DIM((PyArrayObject*)coords, 1) != 3 ||
        PyArray_SIZE((PyArrayObject*)lat) != 9 ||
        PyArray_SIZE((PyArrayObject*)types_in) != PyArray_DIM((PyArrayObject*)coords, 0))
        return fail(PyExc_TypeError, "expected lattice[3,3], types[N], coords[N,3]");
    // the reference reads the raw buffers (C order); make that explicit instead of assuming it
    PyArrayObject* c_lat = (PyArrayObject*)PyArray_FROM_OTF(lat, ft, NPY_ARRAY_IN_ARRAY);
    PyArrayObject* c_coords = (PyArrayObject*)PyArray_FROM_OTF(coords, ft, NPY_ARRAY_IN_ARRAY);
    PyArrayObject* c_types = (PyArrayObject*)PyArray_FROM_OTF(types_in, NPY_INT32, NPY_ARRAY_IN_ARRAY | NPY_ARRAY_FORCECAST);
    if (!c_lat || !c_coords || !c_types) {
        Py_XDECREF(c_lat); Py_XDECREF(c_coords); Py_XDECREF(c_types);
        return nullptr;
    }
    int pbc_i[3];
    for (int i = 0; i < 3; i++) pbc_i[i] = PyObject_IsTrue(PyList_GetItem(pbc, i)) ? 1 : 0;
    const long umax_l = PyLong_AsLong(umax);
    PyObject* out;
    if (umax_l <= 0 || umax_l > (1 << 20)) out = fail(PyExc_RuntimeError, "umax must be positive");
    else
        out = run(c_lat, c_types, c_coords, PyFloat_AsDouble(rcut), (int)umax_l, PyObject_IsTrue(is_cart), pbc_i,
                  PyObject_IsTrue(sort), ft);
    Py_DECREF(c_lat); Py_DECREF(c_coords); Py_DECREF(c_types);
    return out;
}

PyMethodDef methods[] = {
    {"find_info4mlff", (PyCFunction)&py_find_info4mlff, METH_VARARGS, "nblist.find_info4mlff() on the GPU"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef moddef = {PyModuleDef_HEAD_INIT, "nblist", "periodic neighbour list (libai2pot_hip)", -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit_nblist(void)
{
    import_array();
    return PyModule_Create(&moddef);
}
