/*
 * gapx._pack: gather a Python list of structures into packed arrays.
 *
 *     gather(structures, natoms, species, lat, pos) -> atoms or None
 *
 * structures is a list of dicts with numpy arrays "species" (int32 [n]), "lat"
 * (float64 [3, 3]) and "pos" (float64 [n, 3]), all C-contiguous and aligned;
 * natoms and species (int32), lat and pos (float64) are output arrays.
 * Returns the number of atoms; when it exceeds the outputs' room (species n,
 * pos 3 n), only natoms and lat are written and the caller enlarges them.
 * Returns None, having promised nothing, for any other form: the caller
 * then packs with numpy.  (numpy's concatenate and stack cost 100 to 400 ns
 * per array: 1.2 ms for 2000 structures, against about 0.1 ms here.)
 */
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#define NPY_NO_DEPRECATED_API NPY_1_7_API_VERSION
#include <numpy/arrayobject.h>

static PyObject *k_species, *k_lat, *k_pos;

/* The array v when it is a behaved numpy array of this type and shape. */
static PyArrayObject *plain(PyObject *v, int type, int nd, npy_intp d0, npy_intp d1) {
  if (!v || !PyArray_CheckExact(v)) return NULL;
  PyArrayObject *a = (PyArrayObject *)v;
  if (PyArray_TYPE(a) != type || PyArray_NDIM(a) != nd || !PyArray_ISCARRAY_RO(a)) return NULL;
  if (d0 >= 0 && PyArray_DIM(a, 0) != d0) return NULL;
  if (nd == 2 && PyArray_DIM(a, 1) != d1) return NULL;
  return a;
}

static PyObject *gather(PyObject *self, PyObject *args) {
  PyObject *list, *o[4];
  (void)self;
  if (!PyArg_ParseTuple(args, "O!OOOO", &PyList_Type, &list, &o[0], &o[1], &o[2], &o[3])) return NULL;
  const int types[4] = {NPY_INT32, NPY_INT32, NPY_DOUBLE, NPY_DOUBLE};
  for (int k = 0; k < 4; ++k)
    if (!PyArray_CheckExact(o[k]) || PyArray_TYPE((PyArrayObject *)o[k]) != types[k] ||
        PyArray_NDIM((PyArrayObject *)o[k]) != 1 || !PyArray_ISCARRAY((PyArrayObject *)o[k])) {
      PyErr_SetString(PyExc_TypeError, "gather: outputs are int32, int32, float64, float64 vectors");
      return NULL;
    }
  const Py_ssize_t n = PyList_GET_SIZE(list);
  if (PyArray_DIM((PyArrayObject *)o[0], 0) < n || PyArray_DIM((PyArrayObject *)o[2], 0) < 9 * n) {
    PyErr_SetString(PyExc_ValueError, "gather: natoms or lat too short");
    return NULL;
  }
  npy_int32 *natoms = PyArray_DATA((PyArrayObject *)o[0]), *species = PyArray_DATA((PyArrayObject *)o[1]);
  double *lat = PyArray_DATA((PyArrayObject *)o[2]), *pos = PyArray_DATA((PyArrayObject *)o[3]);
  const npy_intp room_s = PyArray_DIM((PyArrayObject *)o[1], 0), room_p = PyArray_DIM((PyArrayObject *)o[3], 0);
  npy_intp total = 0;
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject *s = PyList_GET_ITEM(list, i);
    if (!PyDict_CheckExact(s)) Py_RETURN_NONE;
    PyArrayObject *sp = plain(PyDict_GetItemWithError(s, k_species), NPY_INT32, 1, -1, 0);
    if (!sp) {
      if (PyErr_Occurred()) return NULL;
      Py_RETURN_NONE;
    }
    const npy_intp na = PyArray_DIM(sp, 0);
    PyArrayObject *la = plain(PyDict_GetItemWithError(s, k_lat), NPY_DOUBLE, 2, 3, 3);
    PyArrayObject *po = plain(PyDict_GetItemWithError(s, k_pos), NPY_DOUBLE, 2, na, 3);
    if (!la || !po || na > 0x7fffffff - total) {
      if (PyErr_Occurred()) return NULL;
      Py_RETURN_NONE;
    }
    natoms[i] = (npy_int32)na;
    memcpy(lat + 9 * i, PyArray_DATA(la), 9 * sizeof(double));
    if (total + na <= room_s && 3 * (total + na) <= room_p) {
      memcpy(species + total, PyArray_DATA(sp), (size_t)na * sizeof(npy_int32));
      memcpy(pos + 3 * total, PyArray_DATA(po), (size_t)na * 3 * sizeof(double));
    }
    total += na;
  }
  return PyLong_FromSsize_t((Py_ssize_t)total);
}

static PyMethodDef methods[] = {{"gather", gather, METH_VARARGS, "gather(structures, natoms, species, lat, pos)"},
                                {NULL, NULL, 0, NULL}};
static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_pack", NULL, -1, methods, NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit__pack(void) {
  import_array();
  k_species = PyUnicode_InternFromString("species");
  k_lat = PyUnicode_InternFromString("lat");
  k_pos = PyUnicode_InternFromString("pos");
  if (!k_species || !k_lat || !k_pos) return NULL;
  return PyModule_Create(&module);
}
