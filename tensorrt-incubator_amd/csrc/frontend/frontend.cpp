// The Python front end's calls on torch tensors, in native code: checks, output allocation, the current stream and the
// call into the C ABI, without an interpreter frame, a ctypes conversion or a torch.cuda look-up in between.
//
// Why: a call on a small tensor is bound by the host.  One launch costs 2.3 us back to back on this chip, and the same
// call through ctypes and torch's Python API cost 8 us (package functions) to 12 us (`tp`), of which
// torch.cuda.current_stream() alone was 2.9 us and each torch.empty() 1.7 us.  From here amax is 4.5 us, the dynamic quantization 5.5.
//
// Two sets of functions:
//   * the package's functions (softmax, quantize, ...): argument for argument what the Python wrappers of the same names
//     document, positional and with every default filled in by the wrapper; a failed precondition is an AssertionError, an
//     unsupported element type a KeyError, a status of the library the package's MtrtHipError;
//   * `tp_*`: the `tp` functions for the arguments a program passes in its steady state (tp.Tensors whose values are in
//     device memory, a constant scale uploaded by an earlier call).  Every condition the general path checks is checked
//     here too; when one does not hold the answer is NotImplemented and the general path in tp.py runs, which words the
//     error or moves the operands.
// The interpreter lock is released around the calls into the library.
#include <Python.h>

#include <ATen/EmptyTensor.h>
#include <ATen/core/Tensor.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/hip/impl/HIPCachingAllocatorMasqueradingAsCUDA.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include <memory>

#include "mtrt_hip.h"

namespace {

PyObject *g_error_type = nullptr;                      // the package's MtrtHipError

// ---- arguments and results ---------------------------------------------------------------------
bool fail(const char *what) {
  PyErr_SetString(PyExc_AssertionError, what);
  return false;
}

const at::Tensor *tensor(PyObject *o) {
  if (!THPVariable_Check(o)) {
    PyErr_Format(PyExc_TypeError, "expected a torch.Tensor, got %s", Py_TYPE(o)->tp_name);
    return nullptr;
  }
  return &THPVariable_Unpack(o);
}

PyObject *wrap(const at::TensorBase &t) { return THPVariable_Wrap(t); }

bool integer(PyObject *o, int64_t *v) {
  *v = PyLong_AsLongLong(o);
  return !(*v == -1 && PyErr_Occurred());
}
bool integer32(PyObject *o, int32_t *v) {
  int64_t wide;
  if (!integer(o, &wide))
    return false;
  *v = int32_t(wide);
  return true;
}
bool number(PyObject *o, float *v) {
  const double d = PyFloat_AsDouble(o);
  *v = float(d);
  return !(d == -1.0 && PyErr_Occurred());
}

// f32 / f16 / bf16 -> the C ABI's code, anything else -> -1
int32_t float_code(at::ScalarType t) {
  switch (t) {
  case at::ScalarType::Float: return MTRT_F32;
  case at::ScalarType::Half: return MTRT_F16;
  case at::ScalarType::BFloat16: return MTRT_BF16;
  default: return -1;
  }
}
bool float_type(const at::Tensor &t, int32_t *code) {
  *code = float_code(t.scalar_type());
  if (*code >= 0)
    return true;
  PyObject *name = PyUnicode_FromFormat("element type %s is not one of float32, float16, bfloat16", c10::toString(t.scalar_type()));
  PyErr_SetObject(PyExc_KeyError, name);
  Py_XDECREF(name);
  return false;
}

bool dense_on_gpu(const at::Tensor &t) { return t.is_cuda() && t.is_contiguous(); }

// Where a call works: the current device's current stream, and torch's memory on the device of `x`.  The device is asked for once;
// on it a tensor is made straight on torch's allocator (one that the program swapped in among them), elsewhere by torch's own
// function, which changes the device for as long as it allocates.  Per tensor 0.30 us against 0.47, the stream 0.02 against 0.08.
class Place {
public:
  explicit Place(const at::Tensor &x) : device(x.device()), here(x.device().index() == c10::hip::current_device()) {
    stream = reinterpret_cast<mtrt_stream_t>((here ? c10::hip::getCurrentHIPStream(device.index()) : c10::hip::getCurrentHIPStream()).stream());
  }
  at::Tensor empty(at::IntArrayRef shape, at::ScalarType type) const {
    if (here)
      return at::Tensor(at::detail::empty_generic(shape, c10::hip::HIPCachingAllocatorMasqueradingAsCUDA::get(), c10::DispatchKeySet(c10::DispatchKey::CUDA), type, std::nullopt));
    return at::Tensor(at::detail::empty_cuda(shape, type, device, std::nullopt));
  }
  // Scratch memory of a call: back with torch's allocator when the call returns, which hands it only to work that follows on
  // the same stream.
  at::Tensor bytes(int64_t n) const { return empty({n}, at::ScalarType::Byte); }
  // storage for n codes: int8 for MTRT_I8, else bytes; two to a byte for the packed types
  at::Tensor codes(int32_t q_dtype, int64_t n) const {
    const bool packed = q_dtype == MTRT_I4_PACKED || q_dtype == MTRT_F4_PACKED;
    return empty({packed ? (n + 1) / 2 : n}, q_dtype == MTRT_I8 ? at::ScalarType::Char : at::ScalarType::Byte);
  }
  mtrt_stream_t stream;

private:
  c10::Device device;
  bool here;
};

bool check(int32_t status) {
  if (status == MTRT_OK)
    return true;
  PyObject *e = g_error_type ? PyObject_CallFunction(g_error_type, "is", status, mtrt_hip_last_error()) : nullptr;
  if (e) {
    PyErr_SetObject(g_error_type, e);
    Py_DECREF(e);
  } else if (!PyErr_Occurred()) {
    PyErr_Format(PyExc_RuntimeError, "mtrt_hip status %d: %s", status, mtrt_hip_last_error());
  }
  return false;
}

// Runs `call` (-> status) without the interpreter lock; the message of a failure is the calling thread's own.
template <class F>
bool launch(F &&call) {
  int32_t status;
  Py_BEGIN_ALLOW_THREADS
  status = call();
  Py_END_ALLOW_THREADS
  return check(status);
}

// the [d0, d1] view a call works on: as given, or [everything before the last axis, last axis] of t
bool view2d(const at::Tensor &t, PyObject *a, PyObject *b, int64_t *d0, int64_t *d1) {
  if (a != Py_None && b != Py_None)
    return integer(a, d0) && integer(b, d1);
  if (t.dim() == 0) {
    *d0 = *d1 = 1;
    return true;
  }
  *d1 = t.size(-1);
  *d0 = *d1 ? t.numel() / *d1 : 0;
  return true;
}

// A tensor argument that may be None: the tensor itself, or nullptr in *t with no error set.
bool optional_tensor(PyObject *o, const at::Tensor **t) {
  *t = nullptr;
  if (o == Py_None)
    return true;
  *t = tensor(o);
  return *t != nullptr;
}

PyObject *none_or_new(PyObject *given, const at::Tensor &made) {
  if (given != Py_None) {
    Py_INCREF(given);
    return given;
  }
  return wrap(made);
}

PyObject *tuple_of(std::initializer_list<PyObject *> items) {   // steals the references
  PyObject *t = PyTuple_New(Py_ssize_t(items.size()));
  Py_ssize_t i = 0;
  for (PyObject *o : items) {
    if (t)
      PyTuple_SET_ITEM(t, i++, o);
    else
      Py_XDECREF(o);
  }
  return t;
}

bool arity(Py_ssize_t n, Py_ssize_t want, const char *name) {
  if (n == want)
    return true;
  PyErr_Format(PyExc_TypeError, "%s takes %zd positional arguments, got %zd", name, want, n);
  return false;
}

// torch calls may throw (out of memory, an axis that is not there, a bad shape): their exceptions become Python's
#define FRONTEND_TRY try {
#define FRONTEND_CATCH                                                   \
  }                                                                      \
  catch (const c10::OutOfMemoryError &e) {                               \
    PyErr_SetString(THPException_OutOfMemory(), e.what_without_backtrace()); \
    return nullptr;                                                      \
  }                                                                      \
  catch (const c10::IndexError &e) {                                     \
    PyErr_SetString(PyExc_IndexError, e.what_without_backtrace());       \
    return nullptr;                                                      \
  }                                                                      \
  catch (const std::exception &e) {                                      \
    PyErr_SetString(PyExc_RuntimeError, e.what());                       \
    return nullptr;                                                      \
  }

PyObject *THPException_OutOfMemory() {
  static PyObject *type = nullptr;
  if (!type) {
    PyObject *torch = PyImport_ImportModule("torch");
    if (torch) {
      type = PyObject_GetAttrString(torch, "OutOfMemoryError");
      Py_DECREF(torch);
    }
    if (!type) {
      PyErr_Clear();
      return PyExc_RuntimeError;
    }
  }
  return type;
}

// ---- the package's functions -------------------------------------------------------------------
// amax(x, qmax) -> (amax, scale)
PyObject *f_amax(PyObject *, PyObject *const *a, Py_ssize_t n) {
  FRONTEND_TRY
  const at::Tensor *x;
  float qmax;
  int32_t dt;
  if (!arity(n, 2, "amax") || !(x = tensor(a[0])))
    return nullptr;
  if (!dense_on_gpu(*x))
    return fail("x must be a contiguous tensor on the GPU"), nullptr;
  if (!float_type(*x, &dt) || !number(a[1], &qmax))
    return nullptr;
  const Place place(*x);
  // each its own storage: callers resize, save and free one without the other
  const at::Tensor amax = place.empty({}, at::ScalarType::Float), scale = place.empty({}, at::ScalarType::Float);
  const mtrt_stream_t s = place.stream;
  if (!launch([&] {
        return mtrt_hip_amax(s, x->data_ptr(), dt, x->numel(), qmax, static_cast<float *>(amax.data_ptr()), static_cast<float *>(scale.data_ptr()));
      }))
    return nullptr;
  return tuple_of({wrap(amax), wrap(scale)});
  FRONTEND_CATCH
}

// amax_scales(x, qmax, kind, d0, d1, nb) -> (amax, scale)
PyObject *f_amax_scales(PyObject *, PyObject *const *a, Py_ssize_t n) {
  FRONTEND_TRY
  const at::Tensor *x;
  float qmax;
  int32_t dt, kind;
  int64_t d0, d1, nb;
  if (!arity(n, 6, "amax_scales") || !(x = tensor(a[0])))
    return nullptr;
  if (!dense_on_gpu(*x))
    return fail("x must be a contiguous tensor on the GPU"), nullptr;
  if (!float_type(*x, &dt) || !number(a[1], &qmax) || !integer32(a[2], &kind) || !view2d(*x, a[3], a[4], &d0, &d1) || !integer(a[5], &nb))
    return nullptr;
  const int64_t count = kind == MTRT_SCALE_UNIFORM ? 1 : kind == MTRT_SCALE_ROW ? nb : (nb ? d0 / nb * d1 : 0);
  const Place place(*x);
  const at::Tensor amax = place.empty({count < 0 ? 0 : count}, at::ScalarType::Float);
  const at::Tensor scale = place.empty({count < 0 ? 0 : count}, at::ScalarType::Float);
  const mtrt_stream_t s = place.stream;
  if (!launch([&] {
        return mtrt_hip_amax_scales(s, x->data_ptr(), dt, kind, d0, d1, nb, qmax, static_cast<float *>(amax.data_ptr()),
                                    static_cast<float *>(scale.data_ptr()));
      }))
    return nullptr;
  return tuple_of({wrap(amax), wrap(scale)});
  FRONTEND_CATCH
}

// quantize(x, scale, q_dtype, kind, d0, d1, nb, flags, out) -> codes
PyObject *f_quantize(PyObject *, PyObject *const *a, Py_ssize_t n) {
  FRONTEND_TRY
  const at::Tensor *x, *scale, *out;
  int32_t dt, q_dtype, kind, flags;
  int64_t d0, d1, nb;
  if (!arity(n, 9, "quantize") || !(x = tensor(a[0])) || !(scale = tensor(a[1])) || !optional_tensor(a[8], &out))
    return nullptr;
  if (!dense_on_gpu(*x) || !scale->is_cuda() || scale->scalar_type() != at::ScalarType::Float)
    return fail("x must be contiguous and on the GPU, scale float32 on the GPU"), nullptr;
  if (!integer32(a[2], &q_dtype) || !integer32(a[3], &kind) || !view2d(*x, a[4], a[5], &d0, &d1) || !integer(a[6], &nb) ||
      !integer32(a[7], &flags) || !float_type(*x, &dt))
    return nullptr;
  const Place place(*x);
  const at::Tensor q = out ? *out : place.codes(q_dtype, d0 * d1);
  const mtrt_stream_t s = place.stream;
  if (!launch([&] {
        return mtrt_hip_quantize(s, x->data_ptr(), dt, q.data_ptr(), q_dtype, static_cast<const float *>(scale->data_ptr()), kind, d0, d1,
                                 nb, flags);
      }))
    return nullptr;
  return none_or_new(a[8], q);
  FRONTEND_CATCH
}

bool shape_of(PyObject *o, c10::SmallVector<int64_t, 6> *shape) {
  if (PyLong_Check(o)) {
    int64_t v;
    if (!integer(o, &v))
      return false;
    shape->push_back(v);
    return true;
  }
  PyObject *seq = PySequence_Fast(o, "shape must be an integer or a sequence of integers");
  if (!seq)
    return false;
  for (Py_ssize_t i = 0; i < PySequence_Fast_GET_SIZE(seq); ++i) {
    int64_t v;
    if (!integer(PySequence_Fast_GET_ITEM(seq, i), &v)) {
      Py_DECREF(seq);
      return false;
    }
    shape->push_back(v);
  }
  Py_DECREF(seq);
  return true;
}

bool made_or_given(const at::Tensor *out, PyObject *type, PyObject *shape_arg, const Place &place, at::Tensor *y) {
  if (out) {
    *y = *out;
    return true;
  }
  if (!THPDtype_Check(type)) {
    PyErr_SetString(PyExc_TypeError, "expected a torch.dtype");
    return false;
  }
  c10::SmallVector<int64_t, 6> shape;
  if (!shape_of(shape_arg, &shape))
    return false;
  *y = place.empty(shape, reinterpret_cast<THPDtype *>(type)->scalar_type);
  return true;
}

// dequantize(q, scale, q_dtype, out_torch_dtype, shape, kind, d0, d1, nb, out) -> values
PyObject *f_dequantize(PyObject *, PyObject *const *a, Py_ssize_t n) {
  FRONTEND_TRY
  const at::Tensor *q, *scale, *out;
  int32_t dt, q_dtype, kind;
  int64_t d0, d1, nb;
  at::Tensor y;
  if (!arity(n, 10, "dequantize") || !(q = tensor(a[0])) || !(scale = tensor(a[1])) || !optional_tensor(a[9], &out))
    return nullptr;
  if (!dense_on_gpu(*q) || scale->scalar_type() != at::ScalarType::Float)
    return fail("q must be contiguous and on the GPU, scale float32"), nullptr;
  const Place place(*q);
  if (!made_or_given(out, a[3], a[4], place, &y) || !integer32(a[2], &q_dtype) || !integer32(a[5], &kind) ||
      !view2d(y, a[6], a[7], &d0, &d1) || !integer(a[8], &nb) || !float_type(y, &dt))
    return nullptr;
  const mtrt_stream_t s = place.stream;
  if (!launch([&] {
        return mtrt_hip_dequantize(s, q->data_ptr(), q_dtype, y.data_ptr(), dt, static_cast<const float *>(scale->data_ptr()), kind, d0, d1, nb);
      }))
    return nullptr;
  return none_or_new(a[9], y);
  FRONTEND_CATCH
}

// quantize_dequantize(x, scale, q_dtype, kind, d0, d1, nb, flags, q_out, y_out) -> (codes, values)
PyObject *f_quantize_dequantize(PyObject *, PyObject *const *a, Py_ssize_t n) {
  FRONTEND_TRY
  const at::Tensor *x, *scale, *q_out, *y_out;
  int32_t dt, q_dtype, kind, flags;
  int64_t d0, d1, nb;
  if (!arity(n, 10, "quantize_dequantize") || !(x = tensor(a[0])) || !(scale = tensor(a[1])) || !optional_tensor(a[8], &q_out) ||
      !optional_tensor(a[9], &y_out))
    return nullptr;
  if (!dense_on_gpu(*x) || scale->scalar_type() != at::ScalarType::Float)
    return fail("x must be contiguous and on the GPU, scale float32"), nullptr;
  if (!integer32(a[2], &q_dtype) || !integer32(a[3], &kind) || !view2d(*x, a[4], a[5], &d0, &d1) || !integer(a[6], &nb) ||
      !integer32(a[7], &flags) || !float_type(*x, &dt))
    return nullptr;
  const Place place(*x);
  const at::Tensor q = q_out ? *q_out : place.codes(q_dtype, d0 * d1);
  const at::Tensor y = y_out ? *y_out : place.empty(x->sizes(), x->scalar_type());
  const mtrt_stream_t s = place.stream;
  if (!launch([&] {
        return mtrt_hip_quantize_dequantize(s, x->data_ptr(), dt, q.data_ptr(), q_dtype, y.data_ptr(),
                                            static_cast<const float *>(scale->data_ptr()), kind, d0, d1, nb, flags);
      }))
    return nullptr;
  return tuple_of({none_or_new(a[8], q), none_or_new(a[9], y)});
  FRONTEND_CATCH
}

// dynamic_quantize_dequantize(x, q_dtype, qmax, flags, dequantize) -> (codes, values or None, amax, scale)
PyObject *f_dynamic_quantize_dequantize(PyObject *, PyObject *const *a, Py_ssize_t n) {
  FRONTEND_TRY
  const at::Tensor *x;
  float qmax;
  int32_t dt, q_dtype, flags;
  if (!arity(n, 5, "dynamic_quantize_dequantize") || !(x = tensor(a[0])))
    return nullptr;
  if (!dense_on_gpu(*x))
    return fail("x must be a contiguous tensor on the GPU"), nullptr;
  const int back = PyObject_IsTrue(a[4]);
  if (back < 0 || !integer32(a[1], &q_dtype) || !number(a[2], &qmax) || !integer32(a[3], &flags) || !float_type(*x, &dt))
    return nullptr;
  const Place place(*x);
  const at::Tensor amax = place.empty({}, at::ScalarType::Float), scale = place.empty({}, at::ScalarType::Float);
  const at::Tensor q = place.codes(q_dtype, x->numel());
  at::Tensor y;
  if (back)
    y = place.empty(x->sizes(), x->scalar_type());
  const mtrt_stream_t s = place.stream;
  if (!launch([&] {
        return mtrt_hip_dynamic_quantize_dequantize(s, x->data_ptr(), dt, q.data_ptr(), q_dtype, back ? y.data_ptr() : nullptr, x->numel(),
                                                    qmax, static_cast<float *>(amax.data_ptr()), static_cast<float *>(scale.data_ptr()), flags);
      }))
    return nullptr;
  PyObject *y_obj = Py_None;
  if (back)
    y_obj = wrap(y);
  else
    Py_INCREF(Py_None);
  return tuple_of({wrap(q), y_obj, wrap(amax), wrap(scale)});
  FRONTEND_CATCH
}

// dynamic_quantize_rows(x, q_dtype, qmax, flags, want_amax) -> (codes, amax or None, scale)
PyObject *f_dynamic_quantize_rows(PyObject *, PyObject *const *a, Py_ssize_t n) {
  FRONTEND_TRY
  const at::Tensor *x;
  float qmax;
  int32_t dt, q_dtype, flags;
  if (!arity(n, 5, "dynamic_quantize_rows") || !(x = tensor(a[0])))
    return nullptr;
  if (!dense_on_gpu(*x) || x->dim() < 1)
    return fail("x must be a contiguous tensor of at least one dimension on the GPU"), nullptr;
  const int want = PyObject_IsTrue(a[4]);
  if (want < 0 || !integer32(a[1], &q_dtype) || !number(a[2], &qmax) || !integer32(a[3], &flags) || !float_type(*x, &dt))
    return nullptr;
  const int64_t d = x->size(-1), rows = d ? x->numel() / d : 0;
  const Place place(*x);
  const at::Tensor scale = place.empty({rows}, at::ScalarType::Float);
  at::Tensor amax;
  if (want)
    amax = place.empty({rows}, at::ScalarType::Float);
  const at::Tensor q = place.codes(q_dtype, x->numel());
  const mtrt_stream_t s = place.stream;
  if (!launch([&] {
        return mtrt_hip_dynamic_quantize_rows(s, x->data_ptr(), dt, q.data_ptr(), q_dtype, rows, d, qmax,
                                              want ? static_cast<float *>(amax.data_ptr()) : nullptr, static_cast<float *>(scale.data_ptr()), flags);
      }))
    return nullptr;
  PyObject *amax_obj = Py_None;
  if (want)
    amax_obj = wrap(amax);
  else
    Py_INCREF(Py_None);
  return tuple_of({wrap(q), amax_obj, wrap(scale)});
  FRONTEND_CATCH
}

// whether blocks run along the last axis (-1 or rank - 1); any axis but the last two fails, and so does one that a tensor of
// this rank does not have
bool last_axis(PyObject *o, int64_t rank, bool *last) {
  int64_t axis;
  if (!integer(o, &axis))
    return false;
  if (axis != -1 && axis != -2 && axis != rank - 1 && axis != rank - 2)
    return fail("axis must be one of the last two");
  *last = axis == -1 || axis == rank - 1;
  if (rank < (*last ? 1 : 2)) {
    PyErr_Format(PyExc_IndexError, "axis %lld of a tensor of rank %lld", (long long)axis, (long long)rank);
    return false;
  }
  return true;
}

// nvfp4_quantize(x, tensor_amax, axis) -> (codes, block scales)
PyObject *f_nvfp4_quantize(PyObject *, PyObject *const *a, Py_ssize_t n) {
  FRONTEND_TRY
  const at::Tensor *x, *amax;
  int32_t dt;
  bool last;
  if (!arity(n, 3, "nvfp4_quantize") || !(x = tensor(a[0])) || !(amax = tensor(a[1])))
    return nullptr;
  if (!dense_on_gpu(*x) || !amax->is_cuda() || amax->scalar_type() != at::ScalarType::Float)
    return fail("x must be contiguous and on the GPU, tensor_amax float32 on the GPU"), nullptr;
  if (!last_axis(a[2], x->dim(), &last))
    return nullptr;
  const int64_t d1 = x->size(-1), d0 = d1 ? x->numel() / d1 : 0;
  c10::SmallVector<int64_t, 6> shape(x->sizes().begin(), x->sizes().end());
  shape[shape.size() - (last ? 1 : 2)] /= 16;
  const Place place(*x);
  const at::Tensor q = place.empty({x->numel() / 2}, at::ScalarType::Byte);
  const at::Tensor scales = place.empty(shape, at::ScalarType::Byte);
  if (!float_type(*x, &dt))
    return nullptr;
  const mtrt_stream_t s = place.stream;
  if (!launch([&] {
        return mtrt_hip_nvfp4_quantize(s, x->data_ptr(), dt, q.data_ptr(), scales.data_ptr(), static_cast<const float *>(amax->data_ptr()), d0,
                                       d1, last ? 1 : 0);
      }))
    return nullptr;
  return tuple_of({wrap(q), wrap(scales)});
  FRONTEND_CATCH
}

// nvfp4_dequantize(q, scales, tensor_amax, out_torch_dtype, shape, axis) -> values
PyObject *f_nvfp4_dequantize(PyObject *, PyObject *const *a, Py_ssize_t n) {
  FRONTEND_TRY
  const at::Tensor *q, *scales, *amax;
  int32_t dt;
  at::Tensor y;
  if (!arity(n, 6, "nvfp4_dequantize") || !(q = tensor(a[0])) || !(scales = tensor(a[1])) || !(amax = tensor(a[2])))
    return nullptr;
  if (!q->is_cuda() || q->scalar_type() != at::ScalarType::Byte || scales->scalar_type() != at::ScalarType::Byte ||
      amax->scalar_type() != at::ScalarType::Float)
    return fail("q and scales must be uint8, tensor_amax float32, on the GPU"), nullptr;
  int64_t axis;
  const Place place(*q);
  if (!made_or_given(nullptr, a[3], a[4], place, &y) || !integer(a[5], &axis) || !float_type(y, &dt))
    return nullptr;
  const bool last = axis == -1 || axis == y.dim() - 1;
  const int64_t d1 = y.size(-1), d0 = d1 ? y.numel() / d1 : 0;
  const mtrt_stream_t s = place.stream;
  if (!launch([&] {
        return mtrt_hip_nvfp4_dequantize(s, q->data_ptr(), scales->data_ptr(), static_cast<const float *>(amax->data_ptr()), y.data_ptr(), dt,
                                         d0, d1, last ? 1 : 0);
      }))
    return nullptr;
  return wrap(y);
  FRONTEND_CATCH
}

// layernorm(x, gamma, beta, eps, out) -> y
PyObject *f_layernorm(PyObject *, PyObject *const *a, Py_ssize_t n) {
  FRONTEND_TRY
  const at::Tensor *x, *gamma, *beta, *out;
  float eps;
  int32_t dt;
  if (!arity(n, 5, "layernorm") || !(x = tensor(a[0])) || !(gamma = tensor(a[1])) || !(beta = tensor(a[2])) || !number(a[3], &eps) ||
      !optional_tensor(a[4], &out))
    return nullptr;
  if (!dense_on_gpu(*x) || gamma->scalar_type() != x->scalar_type() || beta->scalar_type() != x->scalar_type())
    return fail("x must be contiguous and on the GPU, gamma and beta of its type"), nullptr;
  if (!float_type(*x, &dt))
    return nullptr;
  const int64_t d = x->size(-1), rows = d ? x->numel() / d : 0;
  const Place place(*x);
  const at::Tensor y = out ? *out : place.empty(x->sizes(), x->scalar_type());
  const mtrt_stream_t s = place.stream;
  if (!launch([&] { return mtrt_hip_layernorm(s, x->data_ptr(), gamma->data_ptr(), beta->data_ptr(), y.data_ptr(), dt, rows, d, eps); }))
    return nullptr;
  return none_or_new(a[4], y);
  FRONTEND_CATCH
}

// softmax(x, out) -> y
PyObject *f_softmax(PyObject *, PyObject *const *a, Py_ssize_t n) {
  FRONTEND_TRY
  const at::Tensor *x, *out;
  int32_t dt;
  if (!arity(n, 2, "softmax") || !(x = tensor(a[0])) || !optional_tensor(a[1], &out))
    return nullptr;
  if (!dense_on_gpu(*x))
    return fail("x must be a contiguous tensor on the GPU"), nullptr;
  if (!float_type(*x, &dt))
    return nullptr;
  const int64_t d = x->size(-1), rows = d ? x->numel() / d : 0;
  const Place place(*x);
  const at::Tensor y = out ? *out : place.empty(x->sizes(), x->scalar_type());
  const mtrt_stream_t s = place.stream;
  if (!launch([&] { return mtrt_hip_softmax(s, x->data_ptr(), y.data_ptr(), dt, rows, d); }))
    return nullptr;
  return none_or_new(a[1], y);
  FRONTEND_CATCH
}

// gemm_w8a8(a, w_nk, a_scale, w_scale, out) and gemm_w8a8_fragments(a, w_frag, a_scale, w_scale, N, out) -> y
PyObject *w8a8(const at::Tensor &x, const at::Tensor &w, const at::Tensor &as, const at::Tensor &ws, int64_t N, PyObject *given,
               bool fragments) {
  const at::Tensor *out;
  if (!optional_tensor(given, &out))
    return nullptr;
  const int64_t M = x.size(0), K = x.size(1);
  if (as.numel() != M || ws.numel() != N || (fragments ? w.numel() != mtrt_hip_gemm_w8a8_fragments_bytes(K, N) : w.size(1) != K))
    return fail("operand extents do not agree"), nullptr;
  const Place place(x);
  const at::Tensor y = out ? *out : place.empty({M, N}, at::ScalarType::Half);
  const mtrt_stream_t s = place.stream;
  const float *asp = static_cast<const float *>(as.data_ptr()), *wsp = static_cast<const float *>(ws.data_ptr());
  const int64_t scratch_bytes = fragments ? mtrt_hip_gemm_w8a8_fragments_workspace(M, K, N) : 0;
  const at::Tensor scratch = scratch_bytes ? place.bytes(scratch_bytes) : at::Tensor();
  if (!launch([&] {
        return fragments ? mtrt_hip_gemm_w8a8_fragments_ws(s, x.data_ptr(), w.data_ptr(), asp, wsp, y.data_ptr(), M, K, N,
                                                           scratch_bytes ? scratch.data_ptr() : nullptr, scratch_bytes)
                         : mtrt_hip_gemm_w8a8(s, x.data_ptr(), w.data_ptr(), asp, wsp, y.data_ptr(), M, K, N);
      }))
    return nullptr;
  return none_or_new(given, y);
}
PyObject *f_gemm_w8a8(PyObject *, PyObject *const *a, Py_ssize_t n) {
  FRONTEND_TRY
  const at::Tensor *x, *w, *as, *ws;
  if (!arity(n, 5, "gemm_w8a8") || !(x = tensor(a[0])) || !(w = tensor(a[1])) || !(as = tensor(a[2])) || !(ws = tensor(a[3])))
    return nullptr;
  if (!dense_on_gpu(*x) || x->scalar_type() != at::ScalarType::Char || x->dim() != 2 || !w->is_contiguous() ||
      w->scalar_type() != at::ScalarType::Char || w->dim() != 2 || as->scalar_type() != at::ScalarType::Float ||
      ws->scalar_type() != at::ScalarType::Float)
    return fail("a and w_nk must be contiguous int8 matrices on the GPU, the scales float32"), nullptr;
  return w8a8(*x, *w, *as, *ws, w->size(0), a[4], false);
  FRONTEND_CATCH
}
PyObject *f_gemm_w8a8_fragments(PyObject *, PyObject *const *a, Py_ssize_t n) {
  FRONTEND_TRY
  const at::Tensor *x, *w, *as, *ws;
  int64_t N;
  if (!arity(n, 6, "gemm_w8a8_fragments") || !(x = tensor(a[0])) || !(w = tensor(a[1])) || !(as = tensor(a[2])) || !(ws = tensor(a[3])) ||
      !integer(a[4], &N))
    return nullptr;
  if (!dense_on_gpu(*x) || x->scalar_type() != at::ScalarType::Char || x->dim() != 2 || w->scalar_type() != at::ScalarType::Char ||
      as->scalar_type() != at::ScalarType::Float || ws->scalar_type() != at::ScalarType::Float)
    return fail("a must be a contiguous int8 matrix on the GPU, w_frag int8, the scales float32"), nullptr;
  return w8a8(*x, *w, *as, *ws, N, a[5], true);
  FRONTEND_CATCH
}

// gemm_w4a16(a, scale, K, N, block, w_kn_packed, w_prepacked, out) -> y
PyObject *f_gemm_w4a16(PyObject *, PyObject *const *a, Py_ssize_t n) {
  FRONTEND_TRY
  const at::Tensor *x, *scale, *packed, *prepacked, *out;
  int64_t K, N, block;
  if (!arity(n, 8, "gemm_w4a16") || !(x = tensor(a[0])) || !(scale = tensor(a[1])) || !integer(a[2], &K) || !integer(a[3], &N) ||
      !integer(a[4], &block) || !optional_tensor(a[5], &packed) || !optional_tensor(a[6], &prepacked) || !optional_tensor(a[7], &out))
    return nullptr;
  if (!dense_on_gpu(*x) || x->scalar_type() != at::ScalarType::Half || x->dim() < 1 || scale->scalar_type() != at::ScalarType::Half)
    return fail("a must be contiguous float16 on the GPU, scale float16"), nullptr;
  const int64_t M = x->size(0);
  const Place place(*x);
  const at::Tensor y = out ? *out : place.empty({M, N}, at::ScalarType::Half);
  const mtrt_stream_t s = place.stream;
  const int64_t scratch_bytes = prepacked ? mtrt_hip_gemm_w4a16_workspace(M, K, N, block) : 0;
  const at::Tensor scratch = scratch_bytes ? place.bytes(scratch_bytes) : at::Tensor();
  if (!launch([&] {
        return mtrt_hip_gemm_w4a16_ws(s, x->data_ptr(), packed ? packed->data_ptr() : nullptr, prepacked ? prepacked->data_ptr() : nullptr,
                                      scale->data_ptr(), y.data_ptr(), M, K, N, block, scratch_bytes ? scratch.data_ptr() : nullptr,
                                      scratch_bytes);
      }))
    return nullptr;
  return none_or_new(a[7], y);
  FRONTEND_CATCH
}

// linear_dense(x, w_nk, bias, out) -> y
PyObject *f_linear_dense(PyObject *, PyObject *const *a, Py_ssize_t n) {
  FRONTEND_TRY
  const at::Tensor *x, *w, *bias, *out;
  int32_t dt;
  if (!arity(n, 4, "linear_dense") || !(x = tensor(a[0])) || !(w = tensor(a[1])) || !optional_tensor(a[2], &bias) ||
      !optional_tensor(a[3], &out))
    return nullptr;
  if (!dense_on_gpu(*x) || x->dim() != 2 || !w->is_contiguous() || w->dim() != 2 || w->scalar_type() != x->scalar_type())
    return fail("x must be a contiguous matrix on the GPU, w_nk a contiguous matrix of its type"), nullptr;
  const int64_t M = x->size(0), K = x->size(1), N = w->size(0);
  if (w->size(1) != K || (bias && (bias->scalar_type() != x->scalar_type() || bias->numel() != N || !bias->is_contiguous())))
    return fail("operand extents or types do not agree"), nullptr;
  if (!float_type(*x, &dt))
    return nullptr;
  const Place place(*x);
  const at::Tensor y = out ? *out : place.empty({M, N}, x->scalar_type());
  const mtrt_stream_t s = place.stream;
  if (!launch([&] {
        return mtrt_hip_linear_dense(s, x->data_ptr(), w->data_ptr(), bias ? bias->data_ptr() : nullptr, y.data_ptr(), dt, M, K, N);
      }))
    return nullptr;
  return none_or_new(a[3], y);
  FRONTEND_CATCH
}

// ---- tp ----------------------------------------------------------------------------------------
// What tp.py hands over once: its Tensor class and its dtype objects (told apart by identity).
struct TpDtype {
  PyObject *object;
  int32_t code;                                        // the C ABI's element type
  at::ScalarType storage;
};
PyTypeObject *g_tensor = nullptr;
TpDtype g_dtypes[6];                                   // float32, float16, bfloat16, int8, int4, float8
PyObject *s_t, *s_dtype, *s_constant, *s_f32_dev, *g_no_args;

const TpDtype *tp_dtype(PyObject *o) {
  for (const TpDtype &d : g_dtypes)
    if (d.object == o)
      return &d;
  return nullptr;
}
bool is_float(const TpDtype *d) { return d && d < g_dtypes + 3; }
bool is_code(const TpDtype *d) { return d && d >= g_dtypes + 3; }

struct TpTensor {
  const at::Tensor *t = nullptr;
  const TpDtype *dtype = nullptr;
  PyObject *hold_t = nullptr;
  ~TpTensor() { Py_XDECREF(hold_t); }
  // false (no error set): not a tp.Tensor of a known dtype
  bool read(PyObject *o) {
    if (Py_TYPE(o) != g_tensor)
      return false;
    PyObject *d = PyObject_GetAttr(o, s_dtype);
    if (d) {
      dtype = tp_dtype(d);
      Py_DECREF(d);
      hold_t = PyObject_GetAttr(o, s_t);
    }
    if (!hold_t) {
      PyErr_Clear();
      return false;
    }
    if (!dtype || !THPVariable_Check(hold_t))
      return false;
    t = &THPVariable_Unpack(hold_t);
    return t->scalar_type() == dtype->storage;
  }
};

PyObject *not_here() { Py_RETURN_NOTIMPLEMENTED; }

// tp.Tensor(t, _produced=True, _tp_dtype=dtype)
PyObject *produced(const at::Tensor &t, const TpDtype *dtype) {
  PyObject *value = wrap(t);
  PyObject *o = value ? g_tensor->tp_new(g_tensor, g_no_args, nullptr) : nullptr;
  if (o && (PyObject_SetAttr(o, s_t, value) < 0 || PyObject_SetAttr(o, s_dtype, dtype->object) < 0 ||
            PyObject_SetAttr(o, s_constant, Py_False) < 0))
    Py_CLEAR(o);
  Py_XDECREF(value);
  return o;
}

// A constant scale: its f32 copy on the device (kept on the scale by tp._scale_on_device, with the version of the constant that
// it was made from) and the addressing that its rank and `dim` give over `shape`, by the rules of tp.check_qdq_args and
// tp._scale_addressing; false when anything is not as those want it.
struct Scale {
  PyObject *hold = nullptr;
  const at::Tensor *dev = nullptr;
  int32_t kind = 0;
  int64_t d0 = 0, d1 = 0, nb = 1;
  ~Scale() { Py_XDECREF(hold); }
  bool read(PyObject *o, const TpDtype *want, const TpDtype *quantized, at::IntArrayRef shape, PyObject *dim_arg) {
    TpTensor s;
    if (!s.read(o) || s.dtype != want)
      return false;
    PyObject *constant = PyObject_GetAttr(o, s_constant);
    const bool ok = constant == Py_True;
    Py_XDECREF(constant);
    hold = ok ? PyObject_GetAttr(o, s_f32_dev) : nullptr;
    if (!hold) {
      PyErr_Clear();
      return false;
    }
    if (!PyTuple_Check(hold) || PyTuple_GET_SIZE(hold) != 2 || !THPVariable_Check(PyTuple_GET_ITEM(hold, 1)))
      return false;
    int64_t version;
    if (!integer(PyTuple_GET_ITEM(hold, 0), &version)) {
      PyErr_Clear();
      return false;
    }
    if (version != (s.t->is_inference() ? -1 : int64_t(s.t->_version())))
      return false;
    dev = &THPVariable_Unpack(PyTuple_GET_ITEM(hold, 1));
    const int64_t rank = int64_t(shape.size()), srank = s.t->dim();
    int64_t numel = 1;
    for (int64_t e : shape)
      numel *= e;
    if (numel == 0)
      return false;
    if (dim_arg != Py_None) {
      if (!PyLong_Check(dim_arg) || srank != 1)
        return false;
      int64_t dim;
      if (!integer(dim_arg, &dim)) {
        PyErr_Clear();
        return false;
      }
      if (dim < -rank || dim >= rank)
        return false;
      dim = dim < 0 ? dim + rank : dim;
      const int64_t c = shape[size_t(dim)];
      if (s.t->size(0) != c)
        return false;
      int64_t inner = 1;
      for (int64_t i = dim + 1; i < rank; ++i)
        inner *= shape[size_t(i)];
      kind = inner == 1 ? MTRT_SCALE_COL : MTRT_SCALE_ROW;
      d0 = inner == 1 ? numel / c : numel / inner;
      d1 = inner == 1 ? c : inner;
      nb = inner == 1 ? d0 : c;
      return true;
    }
    if (srank == 2) {
      if (rank != 2 || quantized != g_dtypes + 4)      // int4 only
        return false;
      const int64_t s0 = s.t->size(0);
      if (s.t->size(1) != shape[1] || s0 == 0 || shape[0] % s0 != 0)
        return false;
      kind = MTRT_SCALE_COL;
      d0 = shape[0];
      d1 = shape[1];
      nb = d0 / s0;
      return true;
    }
    if (srank != 0)
      return false;
    kind = MTRT_SCALE_UNIFORM;
    d1 = rank ? shape[size_t(rank - 1)] : 1;
    d0 = numel / d1;
    return true;
  }
};

// tp_quantize(input, scale, dtype, dim) / tp_dequantize(...)
template <bool QUANTIZE>
PyObject *f_tp_qdq(PyObject *, PyObject *const *a, Py_ssize_t n) {
  FRONTEND_TRY
  TpTensor in;
  Scale scale;
  if (!arity(n, 4, "tp_quantize / tp_dequantize"))
    return nullptr;
  const TpDtype *target = tp_dtype(a[2]);
  if (!g_tensor || !in.read(a[0]) || !(QUANTIZE ? is_float(in.dtype) && is_code(target) : is_code(in.dtype) && is_float(target)) ||
      !dense_on_gpu(*in.t) ||
      !scale.read(a[1], QUANTIZE ? in.dtype : target, QUANTIZE ? target : in.dtype, in.t->sizes(), a[3]))
    return not_here();
  const Place place(*in.t);
  const at::Tensor out = place.empty(in.t->sizes(), target->storage);
  const float *sp = static_cast<const float *>(scale.dev->data_ptr());
  const mtrt_stream_t s = place.stream;
  if (!launch([&] {
        return QUANTIZE ? mtrt_hip_quantize(s, in.t->data_ptr(), in.dtype->code, out.data_ptr(), target->code, sp, scale.kind, scale.d0,
                                            scale.d1, scale.nb, 0)
                        : mtrt_hip_dequantize(s, in.t->data_ptr(), in.dtype->code, out.data_ptr(), target->code, sp, scale.kind, scale.d0,
                                              scale.d1, scale.nb);
      }))
    return nullptr;
  return produced(out, target);
  FRONTEND_CATCH
}

// tp_layernorm(input, weight, bias, eps)
PyObject *f_tp_layernorm(PyObject *, PyObject *const *a, Py_ssize_t n) {
  FRONTEND_TRY
  TpTensor x, w, b;
  float eps;
  if (!arity(n, 4, "tp_layernorm"))
    return nullptr;
  if (!g_tensor || !x.read(a[0]) || !w.read(a[1]) || !b.read(a[2]) || !is_float(x.dtype) || w.dtype != x.dtype || b.dtype != x.dtype)
    return not_here();
  const int64_t lead = x.t->dim() - w.t->dim();
  if (x.t->dim() < 2 || lead < 0 || !w.t->sizes().equals(x.t->sizes().slice(size_t(lead))) || !w.t->sizes().equals(b.t->sizes()) ||
      !dense_on_gpu(*x.t) || !dense_on_gpu(*w.t) || !dense_on_gpu(*b.t))
    return not_here();
  if (!number(a[3], &eps))
    return nullptr;
  const int64_t d = w.t->numel(), rows = d ? x.t->numel() / d : 0;
  const Place place(*x.t);
  const at::Tensor y = place.empty(x.t->sizes(), x.dtype->storage);
  const mtrt_stream_t s = place.stream;
  if (!launch([&] { return mtrt_hip_layernorm(s, x.t->data_ptr(), w.t->data_ptr(), b.t->data_ptr(), y.data_ptr(), x.dtype->code, rows, d, eps); }))
    return nullptr;
  return produced(y, x.dtype);
  FRONTEND_CATCH
}

// tp_softmax(input, dim): over the last of at least two dimensions
PyObject *f_tp_softmax(PyObject *, PyObject *const *a, Py_ssize_t n) {
  FRONTEND_TRY
  TpTensor x;
  int64_t dim;
  if (!arity(n, 2, "tp_softmax"))
    return nullptr;
  if (!g_tensor || !PyLong_Check(a[1]) || !x.read(a[0]) || !is_float(x.dtype) || !dense_on_gpu(*x.t) || x.t->dim() < 2)
    return not_here();
  if (!integer(a[1], &dim)) {
    PyErr_Clear();
    return not_here();
  }
  if (dim != -1 && dim != x.t->dim() - 1)
    return not_here();
  const int64_t d = x.t->size(-1), rows = d ? x.t->numel() / d : 0;
  const Place place(*x.t);
  const at::Tensor y = place.empty(x.t->sizes(), x.dtype->storage);
  const mtrt_stream_t s = place.stream;
  if (!launch([&] { return mtrt_hip_softmax(s, x.t->data_ptr(), y.data_ptr(), x.dtype->code, rows, d); }))
    return nullptr;
  return produced(y, x.dtype);
  FRONTEND_CATCH
}

// The prepared weight side of a tp.Linear: the operands of mtrt_hip_linear, and the parameter objects and versions they were
// made from.
struct LinearPlan {
  mtrt_hip_linear_plan plan{};
  at::Tensor w, w_frag, w_scale, x_scale;
  at::ScalarType type;
  const TpDtype *dtype;
  PyObject *owners[3];                                 // weight, weight_scale, input_scale (what the module held)
  int64_t versions[3];
  PyObject *options[2];                                // quant_dtype, weight_quant_dim
};
constexpr const char *kPlanName = "mtrt_frontend.LinearPlan";
PyObject *s_weight, *s_weight_scale, *s_input_scale, *s_quant_dtype, *s_quant_dim, *s_native_plan, *s_bias;

// The version of a parameter's storage, as tp.Linear._prepared takes it: of every tp.Tensor, instances of subclasses and of
// other types than their storage's among them (TpTensor::read wants the exact class and would answer "none" then and now).
int64_t version_of(PyObject *o) {
  if (!o || !g_tensor || !PyObject_TypeCheck(o, g_tensor))
    return -1;
  const std::unique_ptr<PyObject, void (*)(PyObject *)> t(PyObject_GetAttr(o, s_t), [](PyObject *held) { Py_XDECREF(held); });
  if (!t)
    PyErr_Clear();
  return t && THPVariable_Check(t.get()) ? int64_t(THPVariable_Unpack(t.get())._version()) : -1;
}

// linear_plan(module, route, q_dtype or None, K, N, w, w_frag, w_scale, x_scale) -> what tp_linear reads from the module's
// _native_plan; the tensors are None or lie contiguous on the GPU
PyObject *f_linear_plan(PyObject *, PyObject *const *a, Py_ssize_t n) {
  FRONTEND_TRY
  if (!arity(n, 9, "linear_plan"))
    return nullptr;
  auto made = std::make_unique<LinearPlan>();
  const at::Tensor *t[4];
  for (int i = 0; i < 4; ++i) {
    if (!optional_tensor(a[5 + i], &t[i]))
      return nullptr;
    if (t[i] && !dense_on_gpu(*t[i]))
      return fail("a plan's operands must be contiguous and on the GPU"), nullptr;
  }
  mtrt_hip_linear_plan &p = made->plan;
  PyObject *d = PyObject_GetAttr(a[0], s_dtype);
  made->dtype = d ? tp_dtype(d) : nullptr;
  Py_XDECREF(d);
  const TpDtype *q = a[2] == Py_None ? nullptr : tp_dtype(a[2]);
  if (!integer32(a[1], &p.route) || !integer(a[3], &p.K) || !integer(a[4], &p.N))
    return nullptr;
  if (!is_float(made->dtype) || (a[2] != Py_None && !is_code(q)))
    return fail("a plan needs a float dtype and a quantized one or None"), nullptr;
  p.dtype = made->dtype->code;
  p.q_dtype = q ? q->code : -1;
  made->type = made->dtype->storage;
  at::Tensor *held[4] = {&made->w, &made->w_frag, &made->w_scale, &made->x_scale};
  for (int i = 0; i < 4; ++i)
    if (t[i])
      *held[i] = *t[i];
  p.w = t[0] ? t[0]->data_ptr() : nullptr;
  p.w_frag = t[1] ? t[1]->data_ptr() : nullptr;
  p.w_scale = t[2] ? t[2]->data_ptr() : nullptr;
  p.x_scale = t[3] ? static_cast<const float *>(t[3]->data_ptr()) : nullptr;
  PyObject *const names[5] = {s_weight, s_weight_scale, s_input_scale, s_quant_dtype, s_quant_dim};
  PyObject *found[5];
  for (int i = 0; i < 5; ++i)
    if (!(found[i] = PyObject_GetAttr(a[0], names[i]))) {
      while (i-- > 0)
        Py_DECREF(found[i]);
      return nullptr;
    }
  for (int i = 0; i < 3; ++i) {
    made->owners[i] = found[i];
    made->versions[i] = version_of(found[i]);
  }
  made->options[0] = found[3];
  made->options[1] = found[4];
  PyObject *capsule = PyCapsule_New(made.get(), kPlanName, [](PyObject *c) {
    auto *gone = static_cast<LinearPlan *>(PyCapsule_GetPointer(c, kPlanName));
    for (PyObject *o : gone->owners)
      Py_DECREF(o);
    for (PyObject *o : gone->options)
      Py_DECREF(o);
    delete gone;
  });
  if (!capsule) {
    for (PyObject *o : found)
      Py_DECREF(o);
    return nullptr;
  }
  made.release();
  return capsule;
  FRONTEND_CATCH
}

// tp_linear(module, x): the forward pass when the plan is current, x and the bias lie on the GPU in the module's dtype
PyObject *f_tp_linear(PyObject *, PyObject *const *a, Py_ssize_t n) {
  FRONTEND_TRY
  if (!arity(n, 2, "tp_linear"))
    return nullptr;
  struct Attr {
    PyObject *o;
    Attr(PyObject *of, PyObject *name) : o(PyObject_GetAttr(of, name)) {}
    ~Attr() { Py_XDECREF(o); }
  };
  const Attr capsule(a[0], s_native_plan);
  const LinearPlan *lp = capsule.o && PyCapsule_IsValid(capsule.o, kPlanName)
                             ? static_cast<const LinearPlan *>(PyCapsule_GetPointer(capsule.o, kPlanName))
                             : nullptr;
  TpTensor x;
  if (!lp || !x.read(a[1])) {
    PyErr_Clear();
    return not_here();
  }
  PyObject *const names[5] = {s_weight, s_weight_scale, s_input_scale, s_quant_dtype, s_quant_dim};
  for (int i = 0; i < 5; ++i) {
    const Attr now(a[0], names[i]);
    // options are compared by identity: an equal object that is not the same one takes the general path, which compares values
    if (now.o != (i < 3 ? lp->owners[i] : lp->options[i - 3]) || (i < 3 && version_of(now.o) != lp->versions[i])) {
      PyErr_Clear();
      return not_here();
    }
  }
  const Attr dtype(a[0], s_dtype), bias_object(a[0], s_bias);
  if (!dtype.o || !bias_object.o) {
    PyErr_Clear();
    return not_here();
  }
  TpTensor bias;
  const bool has_bias = bias_object.o != Py_None;
  mtrt_hip_linear_plan p = lp->plan;
  if (dtype.o != lp->dtype->object || x.dtype != lp->dtype || !dense_on_gpu(*x.t) || x.t->dim() < 1 || x.t->size(-1) != p.K ||
      (has_bias && (!bias.read(bias_object.o) || bias.dtype != lp->dtype || !dense_on_gpu(*bias.t) || bias.t->dim() != 1 ||
                    bias.t->size(0) != p.N)) ||
      (p.q_dtype < 0 && reinterpret_cast<uintptr_t>(x.t->data_ptr()) % 16 != 0))
    return not_here();
  p.bias = has_bias ? bias.t->data_ptr() : nullptr;
  c10::SmallVector<int64_t, 6> shape(x.t->sizes().begin(), x.t->sizes().end());
  shape.back() = p.N;
  const int64_t M = x.t->numel() / p.K;
  int64_t scratch_bytes = mtrt_hip_linear_workspace(&p, M);
  const Place place(*x.t);
  const at::Tensor y = place.empty(shape, lp->type);
  at::Tensor scratch;
  if (scratch_bytes) {
    try {
      scratch = place.bytes(scratch_bytes);
    } catch (const c10::OutOfMemoryError &) {
      // a float32 product without memory for its partial sums runs unsplit; what it cannot do without is that of an x that is quantized
      const int64_t least = p.dtype != MTRT_F32 ? scratch_bytes : p.q_dtype < 0 ? 0 : (M * p.K * 4 + 255) / 256 * 256;
      if (least >= scratch_bytes)
        throw;
      scratch_bytes = least;
      if (least)
        scratch = place.bytes(least);
    }
  }
  const mtrt_stream_t s = place.stream;
  if (!launch([&] {
        return mtrt_hip_linear(s, &p, x.t->data_ptr(), y.data_ptr(), M, scratch_bytes ? scratch.data_ptr() : nullptr, scratch_bytes);
      }))
    return nullptr;
  return produced(y, lp->dtype);
  FRONTEND_CATCH
}

// ---- set-up --------------------------------------------------------------------------------------
PyObject *f_set_error_type(PyObject *, PyObject *type) {
  Py_INCREF(type);
  Py_XSETREF(g_error_type, type);
  Py_RETURN_NONE;
}

// bind_tp(Tensor, float32, float16, bfloat16, int8, int4, float8)
PyObject *f_bind_tp(PyObject *, PyObject *const *a, Py_ssize_t n) {
  if (!arity(n, 7, "bind_tp"))
    return nullptr;
  if (!PyType_Check(a[0])) {
    PyErr_SetString(PyExc_TypeError, "bind_tp: the first argument is the Tensor class");
    return nullptr;
  }
  static const int32_t codes[] = {MTRT_F32, MTRT_F16, MTRT_BF16, MTRT_I8, MTRT_I4, MTRT_F8E4M3FN};
  static const at::ScalarType types[] = {at::ScalarType::Float, at::ScalarType::Half, at::ScalarType::BFloat16,
                                         at::ScalarType::Char,  at::ScalarType::Char, at::ScalarType::Byte};
  for (int i = 0; i < 6; ++i) {
    Py_INCREF(a[1 + i]);
    g_dtypes[i] = {a[1 + i], codes[i], types[i]};
  }
  Py_INCREF(a[0]);
  g_tensor = reinterpret_cast<PyTypeObject *>(a[0]);
  Py_RETURN_NONE;
}

#define FAST(name, fn) {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(fn)), METH_FASTCALL, nullptr}
PyMethodDef g_methods[] = {
    FAST("amax", f_amax),
    FAST("amax_scales", f_amax_scales),
    FAST("quantize", f_quantize),
    FAST("dequantize", f_dequantize),
    FAST("quantize_dequantize", f_quantize_dequantize),
    FAST("dynamic_quantize_dequantize", f_dynamic_quantize_dequantize),
    FAST("dynamic_quantize_rows", f_dynamic_quantize_rows),
    FAST("nvfp4_quantize", f_nvfp4_quantize),
    FAST("nvfp4_dequantize", f_nvfp4_dequantize),
    FAST("layernorm", f_layernorm),
    FAST("softmax", f_softmax),
    FAST("gemm_w8a8", f_gemm_w8a8),
    FAST("gemm_w8a8_fragments", f_gemm_w8a8_fragments),
    FAST("gemm_w4a16", f_gemm_w4a16),
    FAST("linear_dense", f_linear_dense),
    FAST("tp_quantize", f_tp_qdq<true>),
    FAST("tp_dequantize", f_tp_qdq<false>),
    FAST("tp_layernorm", f_tp_layernorm),
    FAST("tp_softmax", f_tp_softmax),
    FAST("linear_plan", f_linear_plan),
    FAST("tp_linear", f_tp_linear),
    {"set_error_type", f_set_error_type, METH_O, nullptr},
    FAST("bind_tp", f_bind_tp),
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "mtrt_frontend", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

} // namespace

PyMODINIT_FUNC PyInit_mtrt_frontend(void) {
  s_t = PyUnicode_InternFromString("_t");
  s_dtype = PyUnicode_InternFromString("dtype");
  s_constant = PyUnicode_InternFromString("is_cpu_constant");
  s_f32_dev = PyUnicode_InternFromString("_f32_dev");
  g_no_args = PyTuple_New(0);
  s_weight = PyUnicode_InternFromString("weight");
  s_weight_scale = PyUnicode_InternFromString("weight_scale");
  s_input_scale = PyUnicode_InternFromString("input_scale");
  s_quant_dtype = PyUnicode_InternFromString("quant_dtype");
  s_quant_dim = PyUnicode_InternFromString("weight_quant_dim");
  s_native_plan = PyUnicode_InternFromString("_native_plan");
  s_bias = PyUnicode_InternFromString("bias");
  if (!s_t || !s_dtype || !s_constant || !s_f32_dev || !g_no_args || !s_weight || !s_weight_scale || !s_input_scale || !s_quant_dtype ||
      !s_quant_dim || !s_native_plan || !s_bias)
    return nullptr;
  return PyModule_Create(&g_module);
}
