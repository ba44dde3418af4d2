// CPython module behind the operators of the package on torch tensors: the plain case of each - contiguous tensors of
// the documented types on the current device - from the Python call to the launch without going back to Python.  A
// small operator is bound by that way, not by the GPU: through ctypes a call cost 11 us of which the launch is 3.
// Every function returns None for what it leaves to the Python form of the operator (other layouts and ranks, batches,
// mismatches and whatever the library refuses), which carries the checks and raises the errors.
#include <Python.h>

#include <ATen/Functions.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "tfcc_rocm.h"

namespace {

using at::Tensor;

// The caller keeps the reference; nullptr: not a tensor this module takes (one without memory of its own, as inside
// torch.func transforms, is none).
const Tensor* plain(PyObject* o, at::ScalarType type, c10::DeviceIndex device) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const Tensor& t = THPVariable_Unpack(o);
  if (!t.is_cuda() || !t.has_storage() || t.layout() != at::kStrided || t.scalar_type() != type || t.get_device() != device || !t.is_contiguous()) return nullptr;
  return &t;
}

const Tensor* plain_scalar(PyObject* o, c10::DeviceIndex device) {
  const Tensor* t = plain(o, at::kFloat, device);
  return t && t->dim() == 1 && t->numel() == 1 ? t : nullptr;
}

Tensor empty(at::IntArrayRef shape, at::ScalarType type, c10::DeviceIndex device) {
  return at::detail::empty_cuda(shape, type, c10::Device(c10::kCUDA, device), std::nullopt);
}

// The two ends of a range: two tensors over one allocation.  Taking and giving back the second was 0.3 us of a call that the host bounds:
// quantize of 1 x 64 4.8 -> 4.5 us, 1 x 64 x 64 product 5.0 -> 4.7; the four calls of a quantized layer gain 1.5 to 2 % (24.8 -> 24.4, 21 -> 20.4).
struct Range {
  Tensor low, high;
  explicit Range(c10::DeviceIndex device) : low(empty({2}, at::kFloat, device)) {
    high = at::detail::make_tensor<c10::TensorImpl>(c10::Storage(low.storage()), c10::DispatchKeySet(c10::DispatchKey::CUDA), low.dtype());
    high.unsafeGetTensorImpl()->set_storage_offset(1);
    high.unsafeGetTensorImpl()->set_sizes_contiguous({1});
    low.unsafeGetTensorImpl()->set_sizes_contiguous({1});
  }
};

template <class T = void>
T* data(const Tensor* t) { return t ? static_cast<T*>(t->unsafeGetTensorImpl()->mutable_data()) : nullptr; }
template <class T = void>
T* data(const Tensor& t) { return data<T>(&t); }

bool fits(int64_t v) { return v > 0 && v <= 0x7fffffff; }

// the device of the first operand, where that is the current one; -1 (which no GPU tensor has) otherwise
struct Here {
  c10::DeviceIndex device = -1;
  explicit Here(PyObject* first) {
    if (!THPVariable_CheckExact(first) || !THPVariable_Unpack(first).is_cuda()) return;
    const c10::DeviceIndex d = THPVariable_Unpack(first).get_device();
    if (d == c10::hip::current_device()) device = d;
  }
  void* stream() const { return c10::hip::getCurrentHIPStream(device).stream(); }
};

// The launch itself runs without the interpreter lock, as through ctypes.  What is thrown on the way - a data pointer
// that cannot be had, memory of the library's own bookkeeping - becomes a Python error only with the lock held again.
struct Unlocked {
  PyThreadState* state = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(state); }
};
template <class F>
int launch(F&& f) {
  Unlocked unlocked;
  return f();
}

PyObject* wrap(Tensor t) { return THPVariable_Wrap(std::move(t)); }

PyObject* pack(std::initializer_list<PyObject*> items) {
  PyObject* r = PyTuple_New(static_cast<Py_ssize_t>(items.size()));
  Py_ssize_t i = 0;
  for (PyObject* o : items) {
    if (o == nullptr) {
      for (PyObject* p : items) Py_XDECREF(p);
      Py_XDECREF(r);
      return nullptr;
    }
    ++i;
  }
  if (r == nullptr) return nullptr;
  i = 0;
  for (PyObject* o : items) PyTuple_SET_ITEM(r, i++, o);
  return r;
}

PyObject* none() { Py_RETURN_NONE; }

// blas_matmul(a, b, bias or None)
PyObject* blas_matmul(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 3) return none();
  Here here(args[0]);
  const Tensor* a = plain(args[0], at::kFloat, here.device);
  const Tensor* b = plain(args[1], at::kFloat, here.device);
  const Tensor* bias = args[2] == Py_None ? nullptr : plain(args[2], at::kFloat, here.device);
  if (!a || !b || (args[2] != Py_None && !bias)) return none();
  const int64_t ra = a->dim(), rb = b->dim();
  if (ra < 2 || (rb != 2 && rb != ra)) return none();
  const int64_t m = a->size(ra - 2), k = a->size(ra - 1), cols = b->size(rb - 1);
  if (b->size(rb - 2) != k || (bias && (bias->dim() != 1 || bias->size(0) != cols))) return none();
  if (a->numel() == 0 || b->numel() == 0) return none();
  int64_t batch = 1;
  at::DimVector shape(a->sizes().begin(), a->sizes().end());
  for (int64_t i = 0; i + 2 < ra; ++i) {
    if (rb != 2 && b->size(i) != a->size(i)) return none();
    batch *= a->size(i);
  }
  if (!fits(m) || !fits(k) || !fits(cols) || !fits(batch)) return none();
  shape[ra - 1] = cols;
  Tensor out = empty(shape, at::kFloat, here.device);
  const uint64_t sa = ra == 2 && rb != 2 ? 0 : static_cast<uint64_t>(m) * k, sb = rb == 2 && ra != 2 ? 0 : static_cast<uint64_t>(k) * cols;
  void* stream = here.stream();
  if (launch([&] {
        return tfcc_rocm_sgemm_strided_batched(stream, data<float>(a), sa, data<float>(b), sb, data<float>(bias), data<float>(out),
                                               static_cast<uint64_t>(m) * cols, static_cast<unsigned>(m), static_cast<unsigned>(cols),
                                               static_cast<unsigned>(k), static_cast<unsigned>(batch));
      }) != TFCC_ROCM_OK)
    return none();
  return wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// reduce_sum(a, row)
PyObject* reduce_sum(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 2 || !THPVariable_CheckExact(args[0]) || !PyBool_Check(args[1])) return none();
  Here here(args[0]);
  const at::ScalarType type = THPVariable_Unpack(args[0]).scalar_type();
  if (type != at::kByte && type != at::kChar) return none();
  const Tensor* a = plain(args[0], type, here.device);
  if (!a || a->dim() != 2 || !fits(a->size(0)) || !fits(a->size(1))) return none();
  const bool row = args[1] == Py_True;
  const unsigned r = static_cast<unsigned>(a->size(0)), c = static_cast<unsigned>(a->size(1));
  Tensor out = empty({row ? a->size(0) : a->size(1)}, at::kInt, here.device);
  void* stream = here.stream();
  const int code = type == at::kByte ? TFCC_ROCM_U8 : TFCC_ROCM_S8;
  if (launch([&] {
        return (row ? tfcc_rocm_reduce_sum_rows : tfcc_rocm_reduce_sum_cols)(stream, data(a), code, 1, r, c, data<int32_t>(out));
      }) != TFCC_ROCM_OK)
    return none();
  return wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// The descriptor of a 2-D quantized product from the eight leading arguments of both forms below; false: not plain.
bool describe(PyObject* const* args, const Here& here, tfcc_rocm_qgemm_desc& d) {
  const Tensor* a = plain(args[0], at::kByte, here.device);
  const Tensor* ra = plain(args[1], at::kInt, here.device);
  const Tensor *minA = plain_scalar(args[2], here.device), *maxA = plain_scalar(args[3], here.device);
  const Tensor* b = plain(args[4], at::kChar, here.device);
  const Tensor* rb = plain(args[5], at::kInt, here.device);
  const Tensor *minB = plain_scalar(args[6], here.device), *maxB = plain_scalar(args[7], here.device);
  if (!a || !ra || !minA || !maxA || !b || !rb || !minB || !maxB) return false;
  if (a->dim() != 2 || b->dim() != 2 || ra->dim() != 1 || rb->dim() != 1) return false;
  const int64_t m = a->size(0), k = a->size(1), n = b->size(1);
  if (!fits(m) || !fits(k) || !fits(n) || b->size(0) != k || ra->size(0) != m || rb->size(0) != n) return false;
  d.a = data<uint8_t>(a);
  d.b = data<int8_t>(b);
  d.rowsum_a = data<int32_t>(ra);
  d.colsum_b = data<int32_t>(rb);
  d.stride_c = static_cast<uint64_t>(m) * n;
  d.m = static_cast<unsigned>(m);
  d.n = static_cast<unsigned>(n);
  d.k = static_cast<unsigned>(k);
  d.batch = 1;
  d.min_a = data<float>(minA);
  d.max_a = data<float>(maxA);
  d.min_b = data<float>(minB);
  d.max_b = data<float>(maxB);
  return true;
}

// quantization_matmul(a, reduce_a, min_a, max_a, b, reduce_b, min_b, max_b)
PyObject* quantization_matmul(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 8) return none();
  Here here(args[0]);
  tfcc_rocm_qgemm_desc d{};
  if (!describe(args, here, d)) return none();
  Tensor c = empty({d.m, d.n}, at::kInt, here.device);
  Range range(here.device);
  d.min_c = data<float>(range.low);
  d.max_c = data<float>(range.high);
  void* stream = here.stream();
  if (launch([&] { return tfcc_rocm_gemm_u8s8s32(stream, &d, data<int32_t>(c)); }) != TFCC_ROCM_OK) return none();
  return pack({wrap(std::move(c)), wrap(std::move(range.low)), wrap(std::move(range.high))});
  END_HANDLE_TH_ERRORS
}

// quantization_matmul_requantize(... the eight above, min_out, max_out, want_acc, colsum_exact)
PyObject* quantization_matmul_requantize(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 12 || !PyBool_Check(args[10]) || !PyBool_Check(args[11])) return none();
  Here here(args[0]);
  tfcc_rocm_qgemm_desc d{};
  if (!describe(args, here, d)) return none();
  const Tensor *minOut = plain_scalar(args[8], here.device), *maxOut = plain_scalar(args[9], here.device);
  if (!minOut || !maxOut) return none();
  Tensor q = empty({d.m, d.n}, at::kByte, here.device), c;
  Range range(here.device);
  if (args[10] == Py_True) c = empty({d.m, d.n}, at::kInt, here.device);
  d.min_c = data<float>(range.low);
  d.max_c = data<float>(range.high);
  d.colsum_b_is_exact = args[11] == Py_True ? 1 : 0;
  void* stream = here.stream();
  if (launch([&] {
        return tfcc_rocm_gemm_u8s8s32_requant_u8(stream, &d, c.defined() ? data<int32_t>(c) : nullptr, data<uint8_t>(q), 0.0, 0.0, 0.0, 0,
                                                 data<float>(minOut), data<float>(maxOut));
      }) != TFCC_ROCM_OK)
    return none();
  PyObject* acc = c.defined() ? wrap(std::move(c)) : none();
  return pack({wrap(std::move(q)), acc, wrap(std::move(range.low)), wrap(std::move(range.high))});
  END_HANDLE_TH_ERRORS
}

struct Skinny {
  const Tensor *a, *ra, *rb, *scale;
  int32_t offsetA, offsetB;
  float scaleA;
};

bool skinny_offsets(PyObject* oa, PyObject* ob, PyObject* sa, Skinny& s) {
  if (!PyLong_CheckExact(oa) || !PyLong_CheckExact(ob) || !PyFloat_CheckExact(sa)) return false;
  int overflow = 0;
  const long long x = PyLong_AsLongLongAndOverflow(oa, &overflow);
  if (overflow || x < INT32_MIN || x > INT32_MAX) return false;
  const long long y = PyLong_AsLongLongAndOverflow(ob, &overflow);
  if (overflow || y < INT32_MIN || y > INT32_MAX) return false;
  s.offsetA = static_cast<int32_t>(x);
  s.offsetB = static_cast<int32_t>(y);
  s.scaleA = static_cast<float>(PyFloat_AS_DOUBLE(sa));
  return true;
}

bool skinny_tensors(PyObject* a, PyObject* ra, PyObject* rb, PyObject* scale, const Here& here, Skinny& s) {
  s.a = plain(a, at::kByte, here.device);
  s.ra = plain(ra, at::kInt, here.device);
  s.rb = plain(rb, at::kInt, here.device);
  s.scale = plain(scale, at::kFloat, here.device);
  return s.a && s.ra && s.rb && s.scale && s.a->dim() == 2 && fits(s.a->size(0)) && fits(s.a->size(1)) && s.ra->numel() >= s.a->size(0);
}

// gemv_dequant(a, b, reduce_a, reduce_b, offset_a, offset_b, scale_a, scale_b, want_acc, colsum_exact)
PyObject* gemv_dequant(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 10 || !PyBool_Check(args[8]) || !PyBool_Check(args[9])) return none();
  Here here(args[0]);
  Skinny s;
  const Tensor* b = plain(args[1], at::kChar, here.device);
  if (!b || b->dim() != 2 || !skinny_tensors(args[0], args[2], args[3], args[7], here, s) || !skinny_offsets(args[4], args[5], args[6], s)) return none();
  const int64_t m = s.a->size(0), k = s.a->size(1), cols = b->size(1);
  if (b->size(0) != k || !fits(cols) || s.rb->numel() < cols || s.scale->numel() < cols) return none();
  Tensor acc, out = empty({m, cols}, at::kFloat, here.device);
  if (args[8] == Py_True) acc = empty({m, cols}, at::kInt, here.device);
  void* stream = here.stream();
  const unsigned flags = args[9] == Py_True ? TFCC_ROCM_GEMV_COLSUM_B_IS_EXACT : 0;
  if (launch([&] {
        return tfcc_rocm_gemv_u8s8s32_flags(stream, data<uint8_t>(s.a), data<int8_t>(b), data<int32_t>(s.ra), data<int32_t>(s.rb), s.offsetA,
                                            s.offsetB, static_cast<unsigned>(m), static_cast<unsigned>(cols), static_cast<unsigned>(k),
                                            acc.defined() ? data<int32_t>(acc) : nullptr, s.scaleA, data<float>(s.scale), data<float>(out), flags);
      }) != TFCC_ROCM_OK)
    return none();
  PyObject* accObject = acc.defined() ? wrap(std::move(acc)) : none();
  return pack({wrap(std::move(out)), accObject});
  END_HANDLE_TH_ERRORS
}

// gemv_dequant_packed(a, packed, n, reduce_a, reduce_b, offset_a, offset_b, scale_a, scale_b, want_acc)
PyObject* gemv_dequant_packed(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 10 || !PyBool_Check(args[9]) || !PyLong_CheckExact(args[2])) return none();
  Here here(args[0]);
  Skinny s;
  const Tensor* packed = plain(args[1], at::kByte, here.device);
  int overflow = 0;
  const long long cols = PyLong_AsLongLongAndOverflow(args[2], &overflow);
  if (overflow || !fits(cols) || !packed || !skinny_tensors(args[0], args[3], args[4], args[8], here, s) ||
      !skinny_offsets(args[5], args[6], args[7], s))
    return none();
  const int64_t m = s.a->size(0), k = s.a->size(1);
  if (s.rb->numel() < cols || s.scale->numel() < cols ||
      static_cast<size_t>(packed->numel()) < tfcc_rocm_gemv_packed_size(static_cast<unsigned>(cols), static_cast<unsigned>(k)))
    return none();
  Tensor acc, out = empty({m, cols}, at::kFloat, here.device);
  if (args[9] == Py_True) acc = empty({m, cols}, at::kInt, here.device);
  void* stream = here.stream();
  if (launch([&] {
        return tfcc_rocm_gemv_u8s8s32_packed(stream, data<uint8_t>(s.a), data(packed), data<int32_t>(s.ra), data<int32_t>(s.rb), s.offsetA,
                                             s.offsetB, static_cast<unsigned>(m), static_cast<unsigned>(cols), static_cast<unsigned>(k),
                                             acc.defined() ? data<int32_t>(acc) : nullptr, s.scaleA, data<float>(s.scale), data<float>(out));
      }) != TFCC_ROCM_OK)
    return none();
  PyObject* accObject = acc.defined() ? wrap(std::move(acc)) : none();
  return pack({wrap(std::move(out)), accObject});
  END_HANDLE_TH_ERRORS
}

// -1: a type the quantization kernels do not take
int quantized_code(at::ScalarType t) {
  switch (t) {
    case at::kChar: return TFCC_ROCM_S8;
    case at::kByte: return TFCC_ROCM_U8;
    case at::kShort: return TFCC_ROCM_S16;
    case at::kInt: return TFCC_ROCM_S32;
    default: return -1;
  }
}

// quantize(a, out_dtype): the form that takes the range from the data
PyObject* quantize(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 2 || !THPDtype_Check(args[1])) return none();
  Here here(args[0]);
  const at::ScalarType type = reinterpret_cast<THPDtype*>(args[1])->scalar_type;
  const int code = quantized_code(type);
  const Tensor* a = plain(args[0], at::kFloat, here.device);
  if (!a || code < 0 || a->numel() == 0) return none();
  Tensor out = empty(a->sizes(), type, here.device);
  Range range(here.device);
  void* stream = here.stream();
  if (launch([&] {
        return tfcc_rocm_quantize_minmax(stream, data<float>(a), static_cast<uint64_t>(a->numel()), data(out), code, data<float>(range.low),
                                         data<float>(range.high));
      }) != TFCC_ROCM_OK)
    return none();
  return pack({wrap(std::move(out)), wrap(std::move(range.low)), wrap(std::move(range.high))});
  END_HANDLE_TH_ERRORS
}

// dequantize(a, min, max)
PyObject* dequantize(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 3 || !THPVariable_CheckExact(args[0])) return none();
  Here here(args[0]);
  const at::ScalarType type = THPVariable_Unpack(args[0]).scalar_type();
  const int code = quantized_code(type);
  if (code < 0) return none();
  const Tensor* a = plain(args[0], type, here.device);
  const Tensor *lo = plain_scalar(args[1], here.device), *hi = plain_scalar(args[2], here.device);
  if (!a || !lo || !hi || a->numel() == 0) return none();
  Tensor out = empty(a->sizes(), at::kFloat, here.device);
  void* stream = here.stream();
  if (launch([&] {
        return tfcc_rocm_dequantize(stream, data(a), code, static_cast<uint64_t>(a->numel()), data<float>(lo), data<float>(hi), data<float>(out));
      }) != TFCC_ROCM_OK)
    return none();
  return wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

#define TENSOR_CALL(NAME) {#NAME, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(NAME)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {TENSOR_CALL(blas_matmul), TENSOR_CALL(reduce_sum), TENSOR_CALL(quantization_matmul),
                         TENSOR_CALL(quantization_matmul_requantize), TENSOR_CALL(gemv_dequant), TENSOR_CALL(gemv_dequant_packed),
                         TENSOR_CALL(quantize), TENSOR_CALL(dequantize), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_tensor_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__tensor_calls(void) { return PyModule_Create(&module); }
