// The Python calls that are as long as their host side, in one step each: checks, output tensors, current stream, C ABI.
//
// A call of one kernel took 6.6 us through ctypes, of which the launch is 2.8, the C ABI 0.4, torch's new_empty from Python 1.5
// and the rest argument checks and conversions; here the same call takes 4.1.  Every function returns None for a call that it does not
// take (anything but plain contiguous CUDA tensors of the expected types and shapes, a torch mode that wants to see the
// allocation, or no library loaded yet); the Python method then goes its general way, which also raises what there is to raise.  A status other than 0
// comes back as an int.
// The entry points are handed over by address (bind), so that this module works on whichever build of the library is loaded.
#include <ATen/TensorSubclassLikeUtils.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/yscv_hip.h"

namespace {

decltype(&yscv_hip_int4_matmul) p_int4_matmul = nullptr;
decltype(&yscv_hip_int8_matmul) p_int8_matmul = nullptr;
decltype(&yscv_hip_int8_matmul_requant) p_int8_matmul_requant = nullptr;
decltype(&yscv_hip_exec_dql_matmul_integer) p_exec_dql = nullptr;
decltype(&yscv_hip_rms_norm_dev) p_rms_norm = nullptr;
decltype(&yscv_hip_gqa_attention_dev) p_gqa = nullptr;

PyObject *value_name = nullptr;

// a call from before the library was loaded (the general way loads and binds it), or a torch mode
bool not_taken() { return p_gqa == nullptr || at::impl::torch_function_mode_enabled() || c10::impl::dispatch_mode_enabled(); }

// the tensor of a plain CUDA argument, else null
const at::Tensor *plain(PyObject *o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor &t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || !t.is_contiguous() || t.numel() == 0) return nullptr;
  if (t.is_neg() || t.is_conj() || at::isTensorSubclassLike(t)) return nullptr;
  return &t;
}
const at::Tensor *plain_f32(PyObject *o) {
  const at::Tensor *t = plain(o);
  return t && t->scalar_type() == at::kFloat ? t : nullptr;
}

// the pointer inside a handle (ctypes.c_void_p), null for a closed one
void *handle(PyObject *o) {
  if (o == Py_None) return nullptr;
  PyObject *v = PyObject_GetAttr(o, value_name);
  void *p = v && v != Py_None ? PyLong_AsVoidPtr(v) : nullptr;
  Py_XDECREF(v);
  if (PyErr_Occurred()) PyErr_Clear();
  return p;
}

bool as_size(PyObject *o, int64_t &v) {
  v = PyLong_CheckExact(o) ? PyLong_AsLongLong(o) : -1;
  if (PyErr_Occurred()) PyErr_Clear();
  return v > 0;
}

int dtype_code(at::ScalarType t) {
  return t == at::kFloat ? YSCV_HIP_F32 : (t == at::kHalf ? YSCV_HIP_F16 : (t == at::kBFloat16 ? YSCV_HIP_BF16 : -1));
}

// the stream of the current device, as torch.cuda.current_stream() names it
void *stream() { return c10::hip::getCurrentHIPStream().stream(); }

// Other Python threads run meanwhile: the allocator may have to map memory, and the launch may have to wait for the queue.
class NoGil {
 public:
  NoGil() : state_(PyEval_SaveThread()) {}
  ~NoGil() { PyEval_RestoreThread(state_); }  // (an allocation may throw)
  NoGil(const NoGil &) = delete;
  NoGil &operator=(const NoGil &) = delete;

 private:
  PyThreadState *state_;
};

PyObject *result(int32_t st, at::Tensor out) { return st == 0 ? THPVariable_Wrap(std::move(out)) : PyLong_FromLong(st); }

// int4_matmul(handle, x, k, n)
PyObject *int4_matmul(PyObject *, PyObject *const *a, Py_ssize_t na) {
  HANDLE_TH_ERRORS
  int64_t k, n;
  if (na != 4 || not_taken() || !as_size(a[2], k) || !as_size(a[3], n)) Py_RETURN_NONE;
  const at::Tensor *x = plain(a[1]);
  void *w = handle(a[0]);
  if (!x || !w || x->dim() < 1 || x->size(-1) != k) Py_RETURN_NONE;
  const int dt = dtype_code(x->scalar_type());
  if (dt < 0) Py_RETURN_NONE;
  c10::SmallVector<int64_t, 5> shape(x->sizes().begin(), x->sizes().end());
  shape.back() = n;
  const void *xp = x->data_ptr();
  const size_t m = (size_t)(x->numel() / k);
  const at::TensorOptions like = x->options();
  at::Tensor y;
  int32_t st;
  {
    NoGil released;
    y = at::empty(shape, like);
    st = p_int4_matmul(static_cast<const yscv_hip_int4_weight *>(w), xp, dt, y.data_ptr(), dt, m, stream());
  }
  return result(st, std::move(y));
  END_HANDLE_TH_ERRORS
}

// rows of 8-bit integers against a packed B: handle, a, k, n -> null when the call is not taken
const at::Tensor *int8_rows(PyObject *const *a, void *&w, int64_t &k, int64_t &n) {
  if (!as_size(a[2], k) || !as_size(a[3], n)) return nullptr;
  const at::Tensor *t = plain(a[1]);
  w = handle(a[0]);
  if (!t || !w || t->dim() != 2 || t->size(1) != k || (t->scalar_type() != at::kByte && t->scalar_type() != at::kChar)) return nullptr;
  return t;
}

// int8_matmul(handle, a, k, n, a_zp)
PyObject *int8_matmul(PyObject *, PyObject *const *a, Py_ssize_t na) {
  HANDLE_TH_ERRORS
  int64_t k, n;
  void *w;
  if (na != 5 || not_taken() || !PyLong_CheckExact(a[4])) Py_RETURN_NONE;
  const at::Tensor *t = int8_rows(a, w, k, n);
  const long zp = PyLong_AsLong(a[4]);
  if (PyErr_Occurred()) PyErr_Clear();
  if (!t || zp < -128 || zp > 255) Py_RETURN_NONE;
  const void *ap = t->data_ptr();
  const int64_t m = t->size(0);
  const int u8 = t->scalar_type() == at::kByte;
  const at::TensorOptions like = t->options().dtype(at::kInt);
  at::Tensor y;
  int32_t st;
  {
    NoGil released;
    y = at::empty({m, n}, like);
    st = p_int8_matmul(ap, u8, (int32_t)zp, static_cast<const yscv_hip_i8_weight *>(w), (size_t)m, y.data_ptr<int32_t>(), stream());
  }
  return result(st, std::move(y));
  END_HANDLE_TH_ERRORS
}

// int8_requant(handle, a, k, n, a_zp, composite [n] f32, y_zp, round_mode, clamp_lo, clamp_hi)
PyObject *int8_requant(PyObject *, PyObject *const *a, Py_ssize_t na) {
  HANDLE_TH_ERRORS
  int64_t k, n;
  void *w;
  if (na != 10 || not_taken()) Py_RETURN_NONE;
  long v[4];
  const int at_arg[4] = {4, 7, 8, 9};
  for (int i = 0; i < 4; i++) {
    if (!PyLong_CheckExact(a[at_arg[i]])) Py_RETURN_NONE;
    v[i] = PyLong_AsLong(a[at_arg[i]]);
    if (PyErr_Occurred()) PyErr_Clear();
    if (v[i] < -128 || v[i] > 255) Py_RETURN_NONE;
  }
  if (!PyFloat_CheckExact(a[6])) Py_RETURN_NONE;
  const float y_zp = (float)PyFloat_AS_DOUBLE(a[6]);
  const at::Tensor *t = int8_rows(a, w, k, n), *comp = plain_f32(a[5]);
  if (!t || !comp || comp->dim() != 1 || comp->size(0) != n) Py_RETURN_NONE;
  const void *ap = t->data_ptr();
  const float *cp = comp->data_ptr<float>();
  const int64_t m = t->size(0);
  const int u8 = t->scalar_type() == at::kByte;
  const at::TensorOptions like = t->options().dtype(v[2] < 0 ? at::kChar : at::kByte);
  at::Tensor y;
  int32_t st;
  {
    NoGil released;
    y = at::empty({m, n}, like);
    st = p_int8_matmul_requant(ap, u8, (int32_t)v[0], static_cast<const yscv_hip_i8_weight *>(w), (size_t)m, nullptr, cp, 0.0f, y_zp,
                               (int32_t)v[1], (int32_t)v[2], (int32_t)v[3], y.data_ptr(), stream());
  }
  return result(st, std::move(y));
  END_HANDLE_TH_ERRORS
}

// dql_matmul(handle, x, k, n) -> (out, scale, zero point)
PyObject *dql_matmul(PyObject *, PyObject *const *a, Py_ssize_t na) {
  HANDLE_TH_ERRORS
  int64_t k, n;
  if (na != 4 || not_taken() || !as_size(a[2], k) || !as_size(a[3], n)) Py_RETURN_NONE;
  const at::Tensor *x = plain_f32(a[1]);
  void *w = handle(a[0]);
  if (!x || !w || x->dim() != 2 || x->size(1) != k) Py_RETURN_NONE;
  const float *xp = x->data_ptr<float>();
  const int64_t m = x->size(0);
  const at::TensorOptions like = x->options();
  at::Tensor y, scale, zp;
  int32_t st;
  {
    NoGil released;
    y = at::empty({m, n}, like);
    scale = at::empty({1}, like);
    zp = at::empty({1}, like);
    st = p_exec_dql(xp, (size_t)m, static_cast<const yscv_hip_i8_weight *>(w), y.data_ptr<float>(), scale.data_ptr<float>(), zp.data_ptr<float>(), stream());
  }
  if (st != 0) return PyLong_FromLong(st);
  PyObject *t[3] = {THPVariable_Wrap(std::move(y)), THPVariable_Wrap(std::move(scale)), THPVariable_Wrap(std::move(zp))};
  PyObject *r = PyTuple_Pack(3, t[0], t[1], t[2]);
  for (PyObject *o : t) Py_XDECREF(o);
  return r;
  END_HANDLE_TH_ERRORS
}

// rms_norm(x, gamma, eps)
PyObject *rms_norm(PyObject *, PyObject *const *a, Py_ssize_t na) {
  HANDLE_TH_ERRORS
  if (na != 3 || not_taken() || !PyFloat_CheckExact(a[2])) Py_RETURN_NONE;
  const at::Tensor *x = plain_f32(a[0]), *g = plain_f32(a[1]);
  if (!x || !g || x->dim() < 1 || g->dim() != 1 || g->size(0) != x->size(-1)) Py_RETURN_NONE;
  const float eps = (float)PyFloat_AS_DOUBLE(a[2]);
  const size_t d = (size_t)x->size(-1), rows = (size_t)x->numel() / d;
  const float *xp = x->data_ptr<float>(), *gp = g->data_ptr<float>();
  const c10::SmallVector<int64_t, 5> shape(x->sizes().begin(), x->sizes().end());
  const at::TensorOptions like = x->options();
  at::Tensor y;
  int32_t st;
  {
    NoGil released;
    y = at::empty(shape, like);
    st = p_rms_norm(xp, gp, rows, d, eps, y.data_ptr<float>(), stream());
  }
  return result(st, std::move(y));
  END_HANDLE_TH_ERRORS
}

// gqa(q, k, v, heads, kv_heads)
PyObject *gqa(PyObject *, PyObject *const *a, Py_ssize_t na) {
  HANDLE_TH_ERRORS
  int64_t hq, hkv;
  if (na != 5 || not_taken() || !as_size(a[3], hq) || !as_size(a[4], hkv)) Py_RETURN_NONE;
  const at::Tensor *q = plain_f32(a[0]), *k = plain_f32(a[1]), *v = plain_f32(a[2]);
  if (!q || !k || !v || q->dim() != 3 || k->dim() != 3 || v->sizes() != k->sizes()) Py_RETURN_NONE;
  const int64_t B = q->size(0), sq = q->size(1), sk = k->size(1), d = q->size(2) / hq;
  if (k->size(0) != B || k->size(2) != hkv * d || q->size(2) != hq * d) Py_RETURN_NONE;
  const float *qp = q->data_ptr<float>(), *kp = k->data_ptr<float>(), *vp = v->data_ptr<float>();
  const int64_t width = q->size(2);
  const at::TensorOptions like = q->options();
  at::Tensor y;
  int32_t st;
  {
    NoGil released;
    y = at::empty({B, sq, width}, like);
    st = p_gqa(qp, kp, vp, (size_t)B, (size_t)sq, (size_t)sk, (size_t)hq, (size_t)hkv, (size_t)d, y.data_ptr<float>(), stream());
  }
  return result(st, std::move(y));
  END_HANDLE_TH_ERRORS
}

// bind(addresses of the six entry points, in the order of the pointers above)
PyObject *bind(PyObject *, PyObject *const *a, Py_ssize_t na) {
  if (na != 6) {
    PyErr_SetString(PyExc_TypeError, "bind takes six addresses");
    return nullptr;
  }
  void *p[6];
  for (int i = 0; i < 6; i++) {
    p[i] = PyLong_AsVoidPtr(a[i]);
    if (!p[i]) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "bind: null address");
      return nullptr;
    }
  }
  p_int4_matmul = reinterpret_cast<decltype(p_int4_matmul)>(p[0]);
  p_int8_matmul = reinterpret_cast<decltype(p_int8_matmul)>(p[1]);
  p_int8_matmul_requant = reinterpret_cast<decltype(p_int8_matmul_requant)>(p[2]);
  p_exec_dql = reinterpret_cast<decltype(p_exec_dql)>(p[3]);
  p_rms_norm = reinterpret_cast<decltype(p_rms_norm)>(p[4]);
  p_gqa = reinterpret_cast<decltype(p_gqa)>(p[5]);
  Py_RETURN_NONE;
}

// torch.__version__ of the torch whose headers this was built with
PyObject *torch_version(PyObject *, PyObject *) { return PyUnicode_FromString(YSCV_TORCH_VERSION); }

#define YSCV_CALL(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {YSCV_CALL(bind), {"torch_version", torch_version, METH_NOARGS, nullptr}, YSCV_CALL(int4_matmul), YSCV_CALL(int8_matmul), YSCV_CALL(int8_requant),
                         YSCV_CALL(dql_matmul), YSCV_CALL(rms_norm), YSCV_CALL(gqa), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_calls", "The short calls of yscv_amd without ctypes", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__calls() {
  value_name = PyUnicode_InternFromString("value");
  return value_name ? PyModule_Create(&module) : nullptr;
}
