// CPython module behind runtime_api.Model.run: numpy arrays in, numpy arrays out, over the C ABI of
// tfcc_rocm_runtime.h.  Inputs are read where numpy holds them; every output is an array over a block of host memory of
// its own, which goes back with it.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#define NPY_NO_DEPRECATED_API NPY_1_7_API_VERSION
#include <numpy/arrayobject.h>

#include <string>
#include <vector>

#include "tfcc_rocm_runtime.h"

namespace {

// DataType of tfcc_runtime/proto/common.proto:5-20 for a numpy type in native byte order; 0: none
int data_type_of(const PyArray_Descr* d) {
  if (!PyArray_ISNBO(d->byteorder)) return 0;
  const npy_intp size = PyDataType_ELSIZE(d);
  if (d->kind == 'f') return size == 4 ? 1 : size == 8 ? 11 : 0;
  if (d->kind == 'u') return size == 1 ? 2 : size == 2 ? 4 : size == 4 ? 12 : size == 8 ? 13 : 0;
  if (d->kind == 'i') return size == 1 ? 3 : size == 2 ? 5 : size == 4 ? 6 : size == 8 ? 7 : 0;
  return 0;
}

int numpy_type_of(int dtype) {
  switch (dtype) {
    case 1: return NPY_FLOAT32;
    case 2: case 9: return NPY_UINT8;
    case 3: return NPY_INT8;
    case 4: return NPY_UINT16;
    case 5: return NPY_INT16;
    case 6: return NPY_INT32;
    case 7: return NPY_INT64;
    case 11: return NPY_FLOAT64;
    case 12: return NPY_UINT32;
    case 13: return NPY_UINT64;
  }
  return -1;
}

struct Input {
  PyArrayObject* array = nullptr;
  std::string name;
  std::vector<unsigned> shape;
  int dtype = 0;
  Input() = default;
  Input(Input&& o) noexcept : array(o.array), name(std::move(o.name)), shape(std::move(o.shape)), dtype(o.dtype) { o.array = nullptr; }
  ~Input() { Py_XDECREF(array); }
};

bool read_input(PyObject* key, PyObject* value, PyObject* error, Input& in) {
  Py_ssize_t len = 0;
  if (PyUnicode_Check(key)) {
    const char* text = PyUnicode_AsUTF8AndSize(key, &len);
    if (text == nullptr) return false;
    in.name.assign(text, static_cast<size_t>(len));
  } else {
    char* text = nullptr;
    if (PyBytes_AsStringAndSize(key, &text, &len) < 0) return false;
    in.name.assign(text, static_cast<size_t>(len));
  }
  // the C ABI ends a name at its first zero: what follows would be dropped, and another input might answer to the rest
  if (in.name.find('\0') != std::string::npos) {
    PyErr_Format(error, "invalid input name %R", key);
    return false;
  }
  in.array = reinterpret_cast<PyArrayObject*>(PyArray_FromAny(value, nullptr, 0, 0, NPY_ARRAY_C_CONTIGUOUS, nullptr));
  if (in.array == nullptr) return false;
  in.dtype = data_type_of(PyArray_DESCR(in.array));
  if (in.dtype == 0) {
    PyErr_SetObject(PyExc_KeyError, reinterpret_cast<PyObject*>(PyArray_DESCR(in.array)));
    return false;
  }
  const int rank = PyArray_NDIM(in.array);
  if (rank == 0) in.shape.push_back(1);  // a scalar travels as one element
  for (int i = 0; i < rank; ++i) in.shape.push_back(static_cast<unsigned>(PyArray_DIM(in.array, i)));
  return true;
}

void free_result(PyObject* capsule) { tfcc_rocm_runtime_result_free(PyCapsule_GetPointer(capsule, nullptr)); }

PyObject* output_array(const tfcc_rocm_runtime_array& o, PyObject* owner) {
  const int type = numpy_type_of(o.dtype);
  if (type < 0) return PyErr_Format(PyExc_ValueError, "output %s: element type %d", o.name, o.dtype);
  std::vector<npy_intp> dims(o.shape, o.shape + o.rank);
  if (o.bytes == 0) {
    if (dims.empty()) return PyErr_Format(PyExc_ValueError, "output %s has not been set", o.name);
    return PyArray_SimpleNew(static_cast<int>(dims.size()), dims.data(), type);
  }
  PyObject* a = PyArray_SimpleNewFromData(static_cast<int>(dims.size()), dims.data(), type, o.data);
  if (a == nullptr) return nullptr;
  Py_INCREF(owner);
  if (PyArray_SetBaseObject(reinterpret_cast<PyArrayObject*>(a), owner) < 0) {
    Py_DECREF(a);
    return nullptr;
  }
  return a;
}

// run(model handle, {name: array}, exception class) -> {name: array}.  The arrays are read with the interpreter lock
// released: another thread that writes to one meanwhile changes what the run sees.
PyObject* run(PyObject*, PyObject* args) {
  unsigned long long handle = 0;
  PyObject *arrays = nullptr, *error = nullptr;
  if (!PyArg_ParseTuple(args, "KOO", &handle, &arrays, &error)) return nullptr;
  // converting a value may run code of its own, so what is walked is a list; as `for name, a in arrays.items()`, any
  // mapping with such a method will do
  PyObject* pairs = PyDict_CheckExact(arrays) ? PyDict_Items(arrays) : PyObject_CallMethod(arrays, "items", nullptr);
  PyObject* items = pairs ? PySequence_List(pairs) : nullptr;
  Py_XDECREF(pairs);
  if (items == nullptr) return nullptr;
  std::vector<Input> inputs(static_cast<size_t>(PyList_GET_SIZE(items)));
  bool fine = true;
  for (size_t i = 0; i < inputs.size() && fine; ++i) {
    PyObject* item = PySequence_Tuple(PyList_GET_ITEM(items, static_cast<Py_ssize_t>(i)));
    if (item && PyTuple_GET_SIZE(item) != 2) PyErr_SetString(PyExc_ValueError, "items() gives something else than (name, array)");
    fine = item && PyTuple_GET_SIZE(item) == 2 && read_input(PyTuple_GET_ITEM(item, 0), PyTuple_GET_ITEM(item, 1), error, inputs[i]);
    Py_XDECREF(item);
  }
  Py_DECREF(items);
  if (!fine) return nullptr;
  std::vector<tfcc_rocm_runtime_array> views;
  for (Input& in : inputs)
    views.push_back({in.name.c_str(), in.dtype, in.shape.data(), in.shape.size(), PyArray_DATA(in.array),
                     static_cast<size_t>(PyArray_NBYTES(in.array))});
  void* result = nullptr;
  size_t count = 0;
  int status;
  Py_BEGIN_ALLOW_THREADS
  status = tfcc_rocm_runtime_model_run_arrays(reinterpret_cast<void*>(handle), views.data(), views.size(), &result, &count);
  Py_END_ALLOW_THREADS
  if (status != 0) {
    const char* text = tfcc_rocm_runtime_last_error();
    PyObject* message = PyUnicode_DecodeUTF8(text, static_cast<Py_ssize_t>(std::char_traits<char>::length(text)), "replace");
    if (message) PyErr_SetObject(error, message);
    Py_XDECREF(message);
    return nullptr;
  }
  PyObject* outputs = PyDict_New();
  for (size_t i = 0; outputs && i < count; ++i) {
    void* part = nullptr;
    PyObject *owner = nullptr, *a = nullptr;
    if (tfcc_rocm_runtime_result_detach(result, i, &part) != 0) PyErr_NoMemory();
    else if ((owner = PyCapsule_New(part, nullptr, free_result)) == nullptr) tfcc_rocm_runtime_result_free(part);
    if (owner) {
      tfcc_rocm_runtime_array o;
      tfcc_rocm_runtime_result_output(part, 0, &o);
      a = output_array(o, owner);
      if (a == nullptr || PyDict_SetItemString(outputs, o.name, a) < 0) Py_CLEAR(a);
      Py_DECREF(owner);
    }
    if (a == nullptr) Py_CLEAR(outputs);
    Py_XDECREF(a);
  }
  tfcc_rocm_runtime_result_free(result);
  return outputs;
}

PyMethodDef methods[] = {{"run", run, METH_VARARGS, "run(handle, arrays, error) -> {name: ndarray}"}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_model_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__model_calls(void) {
  import_array();
  return PyModule_Create(&module);
}
