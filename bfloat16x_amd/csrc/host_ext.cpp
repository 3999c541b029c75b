// CPython module _host: the per-call host path of the operator wrappers.
//
// A batch-1 GEMV runs a few microseconds on the GPU; checking its tensors in
// Python and converting its 20 arguments through ctypes took about 12 (the
// whole call 15.8 us at 1024x4096, 8.3 us with this module).  Here are
//   gemv(...)       the checks, the output and the launch of ops.bf16x_gemv,
//   plain(...)      the checks of the other wrappers (device, type, layout),
//   stream(device)  torch's current stream,
//   and the hot C-ABI entries with tensors accepted for their pointers.
// gemv and plain only say yes to ordinary tensors that the entry takes as they
// are; on anything else (another type or layout, a wrapped or fake tensor, an
// error) they answer None / False and the wrapper's Python path runs, with its
// conversions and its exceptions.  Nothing is kept between calls.
#include <torch/csrc/autograd/python_variable.h>
#include <c10/hip/HIPStream.h>
#include <ATen/ops/empty.h>

#include <type_traits>
#include <utility>

#include "../../include/bf16x_hip.h"

namespace {

// An ordinary tensor (or Parameter), or null.
const at::Tensor* tensor_of(PyObject* o) { return THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr; }

bool on_gpu(const at::Tensor& t, int device) {
  return t.layout() == c10::kStrided && t.is_cuda() && t.get_device() == device && t.is_contiguous();
}

// The weight's streams in their own types on one GPU: its index, or -1.
int weight_device(PyObject* const* o) {
  static constexpr c10::ScalarType kTypes[4] = {c10::kInt, c10::kInt, c10::kInt, c10::kByte};
  int dev = -1;
  for (int i = 0; i < 4; ++i) {
    const at::Tensor* t = tensor_of(o[i]);
    if (!t || t->scalar_type() != kTypes[i] || !t->is_cuda()) return -1;
    if (i == 0) dev = t->get_device();
    if (!on_gpu(*t, dev)) return -1;
  }
  return dev;
}

int32_t x_code(c10::ScalarType t) {
  return t == c10::kBFloat16 ? BF16X_BF16 : t == c10::kHalf ? BF16X_F16 : t == c10::kFloat ? BF16X_F32 : -1;
}

// The GIL given up for the scope (and taken again when an exception leaves it):
// a launch or an allocation may wait for the GPU, and a host callback that the
// GPU waits for may need Python.
struct WithoutGil {
  PyThreadState* state = PyEval_SaveThread();
  ~WithoutGil() { PyEval_RestoreThread(state); }
};

void* stream_of(int dev) { return (void*)c10::hip::getCurrentHIPStream((c10::DeviceIndex)dev).stream(); }

// gemv(x, sign, mant, delta, emax, tile_off, tile_ent, tile_sat, out_f, in_f,
// sub, out): y; None when the Python path has to take the call; the status (an
// int) when the launch was made and the runtime reports an error
PyObject* gemv(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 12) Py_RETURN_NONE;
  try {
    const int dev = weight_device(a + 1);
    const at::Tensor* x = tensor_of(a[0]);
    if (dev < 0 || !x || !on_gpu(*x, dev) || x_code(x->scalar_type()) < 0) Py_RETURN_NONE;
    const bool exact = a[5] != Py_None;
    const at::Tensor* plan[3] = {nullptr, nullptr, nullptr};
    for (int i = 0; exact && i < 3; ++i) {
      plan[i] = tensor_of(a[5 + i]);
      if (!plan[i] || !plan[i]->is_cuda() || plan[i]->get_device() != dev) Py_RETURN_NONE;
    }
    const int64_t out_f = PyLong_AsLongLong(a[8]), in_f = PyLong_AsLongLong(a[9]);
    const long sub = PyLong_AsLong(a[10]);
    if (PyErr_Occurred()) {
      PyErr_Clear();
      Py_RETURN_NONE;
    }
    if (out_f <= 0 || x->numel() != in_f) Py_RETURN_NONE;
    at::Tensor y;
    if (a[11] != Py_None) {
      const at::Tensor* o = tensor_of(a[11]);
      if (!o || !on_gpu(*o, dev) || o->scalar_type() != c10::kBFloat16 || o->numel() < out_f) Py_RETURN_NONE;
      y = *o;
    }
    const at::Tensor &s = *tensor_of(a[1]), &m = *tensor_of(a[2]), &d = *tensor_of(a[3]), &e = *tensor_of(a[4]);
    auto p = [&](int i) { return exact ? plan[i]->data_ptr() : nullptr; };
    int rc;
    {
      const WithoutGil no_gil;                  // (the caller's references keep the tensors)
      if (!y.defined()) y = at::empty({out_f}, s.options().dtype(c10::kBFloat16));
      rc = bf16x_gemv(x->data_ptr(), x_code(x->scalar_type()), (const int32_t*)s.data_ptr(), s.numel(),
                      (const int32_t*)m.data_ptr(), m.numel(), (const int32_t*)d.data_ptr(), d.numel(),
                      (const uint8_t*)e.data_ptr(), e.numel(), (const uint32_t*)p(0), (const uint32_t*)p(1),
                      (const uint8_t*)p(2), out_f, in_f, (int32_t)sub, exact ? BF16X_EXACT : BF16X_SATURATED,
                      (uint16_t*)y.data_ptr(), stream_of(dev));
    }
    if (rc < 0) Py_RETURN_NONE;                 // refused before the launch
    if (rc > 0) return PyLong_FromLong(rc);     // a runtime error, reported after it: not to be launched again
    return THPVariable_Wrap(std::move(y));
  } catch (...) {
    Py_RETURN_NONE;
  }
}

// plain(x, sign, mant, delta, emax, *more): whether the streams are ordinary
// and x (a bf16, fp16 or fp32 tensor) and the tensors of `more` (None allowed)
// are contiguous on their GPU
PyObject* plain(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n < 5) Py_RETURN_FALSE;
  try {
    const int dev = weight_device(a + 1);
    if (dev < 0) Py_RETURN_FALSE;
    for (Py_ssize_t i = 0; i < n; i = i ? i + 1 : 5) {
      if (i && a[i] == Py_None) continue;
      const at::Tensor* t = tensor_of(a[i]);
      if (!t || !on_gpu(*t, dev) || (i == 0 && x_code(t->scalar_type()) < 0)) Py_RETURN_FALSE;
    }
    Py_RETURN_TRUE;
  } catch (...) {
    Py_RETURN_FALSE;
  }
}

PyObject* stream(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 1) return PyErr_Format(PyExc_TypeError, "stream(device index)");
  const long dev = PyLong_AsLong(a[0]);
  if (dev == -1 && PyErr_Occurred()) return nullptr;
  try {
    return PyLong_FromVoidPtr(stream_of((int)dev));
  } catch (const std::exception& e) {
    return PyErr_Format(PyExc_RuntimeError, "%s", e.what());
  }
}

// One argument of a C entry: an int, or for a pointer a tensor, an address or
// None.  false with a Python error set when it is none of these.
template <class T>
bool from_py(PyObject* o, T& v) {
  if constexpr (std::is_pointer<T>::value) {
    if (o == Py_None) {
      v = nullptr;
      return true;
    }
    if (THPVariable_Check(o)) {
      v = (T)THPVariable_Unpack(o).data_ptr();
      return true;
    }
    v = (T)PyLong_AsVoidPtr(o);
  } else {
    v = (T)PyLong_AsLongLong(o);
  }
  return !PyErr_Occurred();
}

template <class... A, size_t... I>
PyObject* invoke(int (*f)(A...), PyObject* const* a, Py_ssize_t n, std::index_sequence<I...>) {
  if (n != (Py_ssize_t)sizeof...(A)) return PyErr_Format(PyExc_TypeError, "%d arguments expected", (int)sizeof...(A));
  try {
    std::tuple<std::decay_t<A>...> v;
    if (!(from_py(a[I], std::get<I>(v)) && ...)) return nullptr;
    int rc;
    {
      const WithoutGil no_gil;
      rc = f(std::get<I>(v)...);
    }
    return PyLong_FromLong(rc);
  } catch (const std::exception& e) {
    return PyErr_Format(PyExc_RuntimeError, "%s", e.what());
  }
}
template <class... A>
PyObject* invoke(int (*f)(A...), PyObject* const* a, Py_ssize_t n) {
  return invoke(f, a, n, std::index_sequence_for<A...>{});
}

#define ENTRY(name) \
  PyObject* c_##name(PyObject*, PyObject* const* a, Py_ssize_t n) { return invoke(&name, a, n); }
ENTRY(bf16x_decode)
ENTRY(bf16x_gemm)
ENTRY(bf16x_gemm_rows)
ENTRY(bf16x_gemm_chunks)
ENTRY(bf16x_gemm_terms)
ENTRY(bf16x_split_terms)
ENTRY(bf16x_add_terms)
ENTRY(bf16x_gguf_gemv)
ENTRY(bf16x_gguf_gemv_lossless)
ENTRY(bf16x_gguf_gemm)
ENTRY(bf16x_gguf_decode)
ENTRY(bf16x_gguf_decode_lossless)
#undef ENTRY

#define FAST(name, fn) {name, (PyCFunction)(void (*)(void))fn, METH_FASTCALL, nullptr}
#define ENTRY(name) FAST(#name, c_##name)
PyMethodDef methods[] = {FAST("gemv", gemv), FAST("plain", plain), FAST("stream", stream), ENTRY(bf16x_decode),
                         ENTRY(bf16x_gemm), ENTRY(bf16x_gemm_rows), ENTRY(bf16x_gemm_chunks),
                         ENTRY(bf16x_gemm_terms), ENTRY(bf16x_split_terms), ENTRY(bf16x_add_terms), ENTRY(bf16x_gguf_gemv),
                         ENTRY(bf16x_gguf_gemv_lossless), ENTRY(bf16x_gguf_gemm), ENTRY(bf16x_gguf_decode),
                         ENTRY(bf16x_gguf_decode_lossless), {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() { return PyModule_Create(&module); }
