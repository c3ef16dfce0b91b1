// The host's side of a decode call, as an extension module of CPython: what moba_amd/decode.py asks of its tensors, the
// allocation of result and scratch, and the call into libmoba_hip.so.
//
// A decode step of a short conversation is a few microseconds of work for the device (10.1 us a call at 4097 keys, 8
// key/value heads, calls queued one behind the other) and was 21 us for the host: some forty attribute reads, size
// tuples, argument conversions and checks in Python.  Here, with the two launches, it is 11 us: as long as the device
// takes.  (Putting the splits together in the first launch, by its last workgroup, would spare the host the second and
// costs the device more than that: 11.4 us.)
//
// Nothing is kept between calls but the addresses of the library's entry points (bind): types by the library's header, whose
// version the library has to have.  The module itself is tied to one interpreter and one PyTorch: its file name says the
// first, `torch_version` the second, and _lib.host() refuses it for another.  What these functions do not
// take -- tensors that have to be copied first, more sequences than a launch takes -- they leave to the caller.
#include <ATen/ATen.h>
#include <Python.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/moba_hip.h"

namespace {

decltype(&moba_tail_splits) tail_splits = nullptr;
decltype(&moba_tail) tail_call = nullptr;
decltype(&moba_strerror) str_error = nullptr;

constexpr int64_t kHeadDim = 128, kMostSequences = 65535;

const at::Tensor* tensor_of(PyObject* o) { return THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr; }

// q [B,H,q_len,D] and k, v [B,Hkv,Skv,D] that the kernels can take
bool chunk_supported(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v) {
  if (!(q.is_cuda() && k.is_cuda() && v.is_cuda())) return false;
  const auto type = q.scalar_type();
  if ((type != at::kBFloat16 && type != at::kHalf) || k.scalar_type() != type || v.scalar_type() != type) return false;
  if (q.dim() != 4 || k.dim() != 4 || k.sizes() != v.sizes()) return false;
  const auto qs = q.sizes(), ks = k.sizes();
  if (qs[3] != kHeadDim || ks[0] != qs[0] || ks[3] != qs[3] || qs[2] <= 0 || qs[2] > ks[2]) return false;
  return ks[1] > 0 && qs[1] % ks[1] == 0;
}

// ... one token, and 1, 2, 4 or 8 query heads per key/value head
bool supported(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v) {
  if (!chunk_supported(q, k, v) || q.size(2) != 1) return false;
  const int64_t rep = q.size(1) / k.size(1);
  return rep == 1 || rep == 2 || rep == 4 || rep == 8;
}

// The strides of batch, head and token of a tensor that is read where it lies (decode.py: _placed): the stride of a dimension of
// one entry says nothing and is 0.  False for one that has to be copied.
bool in_place(const at::Tensor& t, int64_t row_step, int64_t (&steps)[3]) {
  if (t.dim() != 4) return false;
  const auto size = t.sizes(), stride = t.strides();
  for (int i = 0; i < 3; ++i) steps[i] = size[i] > 1 ? stride[i] : 0;
  return stride[3] == 1 && !((steps[0] | steps[1] | steps[2]) & 7) && steps[2] <= (1 << 23) &&
         ((uintptr_t)t.data_ptr() & 15) == 0 && (stride[2] == row_step || !row_step || size[2] == 1);
}

PyObject* py_supported(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n == 4, "supported(query, key, value, several)");
  const at::Tensor *q = tensor_of(args[0]), *k = tensor_of(args[1]), *v = tensor_of(args[2]);
  TORCH_CHECK_TYPE(q && k && v, "query, key and value must be tensors");
  return PyBool_FromLong(PyObject_IsTrue(args[3]) ? chunk_supported(*q, *k, *v) : supported(*q, *k, *v));
  END_HANDLE_TH_ERRORS
}

// The allocations may have to free memory and the launches wait for room in the queue, where a callback may in turn wait for
// Python: other threads go on meanwhile, as they do under PyTorch's own calls and under ctypes.
struct NoGil {
  PyThreadState* const state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
};

// tail(query, key, value, scaling or None): [B,q_len,H,D] on the decode kernel, or None where that needs copies or pieces
PyObject* py_tail(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n == 4, "tail(query, key, value, scaling)");
  const at::Tensor *qt = tensor_of(args[0]), *kt = tensor_of(args[1]), *vt = tensor_of(args[2]);
  TORCH_CHECK_TYPE(qt && kt && vt, "query, key and value must be tensors");
  TORCH_CHECK(tail_call, "the library's entry points are not bound");
  const at::Tensor &q = *qt, &k = *kt, &v = *vt;
  if (!chunk_supported(q, k, v)) Py_RETURN_NONE;
  double scale = 0.08838834764831845;  // 128 ** -0.5
  if (args[3] != Py_None) {
    scale = PyFloat_AsDouble(args[3]);
    if (PyErr_Occurred()) return nullptr;
  }
  const int64_t b = q.size(0), h = q.size(1), q_len = q.size(2), hkv = k.size(1), skv = k.size(2);
  int64_t qs[3], ks[3], vs[3];
  if (b < 1 || b > kMostSequences || !in_place(q, 0, qs) || !in_place(k, kHeadDim, ks) || !in_place(v, kHeadDim, vs) ||
      ks[0] != vs[0] || ks[1] != vs[1] || ks[2] != vs[2] || skv > INT32_MAX || h > INT32_MAX)
    Py_RETURN_NONE;
  const int splits = tail_splits((int)b, (int)hkv, (int)(h / hkv), (int)q_len, (int)skv);
  const int64_t rows = b * q_len * h * splits;
  const void *const qp = q.const_data_ptr(), *const kp = k.const_data_ptr(), *const vp = v.const_data_ptr();
  const auto type = q.scalar_type();
  const auto device = q.device();
  const int64_t strides[5] = {qs[0], qs[1], qs[2], ks[0], ks[1]};
  at::Tensor out;
  int rc;
  {
    const NoGil no_gil;
    out = at::empty({b, q_len, h, kHeadDim}, at::TensorOptions().dtype(type).device(device));
    // partial outputs, then their log-sum-exps (neither is touched with one split)
    at::Tensor part = at::empty({splits > 1 ? rows * (kHeadDim + 1) : 4}, at::TensorOptions().dtype(at::kFloat).device(device));
    float* const part_o = part.mutable_data_ptr<float>();
    rc = tail_call(qp, kp, vp, out.mutable_data_ptr(), part_o, splits > 1 ? part_o + rows * kHeadDim : part_o, (int)b, (int)h,
                   (int)hkv, (int)q_len, (int)skv, (int)kHeadDim, strides, (float)scale, type == at::kHalf ? 1 : 0,
                   c10::hip::getCurrentHIPStream(device.index()).stream());
  }
  if (rc != 0) {
    PyErr_Format(PyExc_RuntimeError, "moba_tail failed with code %d: %s", rc, str_error(rc));
    return nullptr;
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// in_place(tensor, row_step): the strides of batch, head and token of a [B,heads,tokens,D] tensor that is read where it lies,
// None for one that has to be copied
PyObject* py_in_place(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n == 2 && tensor_of(args[0]), "in_place(tensor, row_step)");
  const int64_t row_step = PyLong_AsLongLong(args[1]);
  if (PyErr_Occurred()) return nullptr;
  int64_t steps[3];
  if (!in_place(*tensor_of(args[0]), row_step, steps)) Py_RETURN_NONE;
  return Py_BuildValue("(LLL)", (long long)steps[0], (long long)steps[1], (long long)steps[2]);
  END_HANDLE_TH_ERRORS
}

// bind(moba_version, moba_tail_splits, moba_tail, moba_strerror): the addresses of the library's entry points
PyObject* py_bind(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n == 4, "bind takes four addresses");
  void* at[4];
  for (int i = 0; i < 4; ++i) {
    at[i] = PyLong_AsVoidPtr(args[i]);
    if (PyErr_Occurred()) return nullptr;
  }
  const int version = reinterpret_cast<decltype(&moba_version)>(at[0])();
  TORCH_CHECK(version == MOBA_ABI_VERSION, "this module was built for version ", MOBA_ABI_VERSION, " of the C ABI, the library has ",
              version);
  tail_splits = reinterpret_cast<decltype(tail_splits)>(at[1]);
  tail_call = reinterpret_cast<decltype(tail_call)>(at[2]);
  str_error = reinterpret_cast<decltype(str_error)>(at[3]);
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"supported", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_supported)), METH_FASTCALL, nullptr},
    {"tail", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_tail)), METH_FASTCALL, nullptr},
    {"in_place", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_in_place)), METH_FASTCALL, nullptr},
    {"bind", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_bind)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() {
  PyObject* const m = PyModule_Create(&module);
  if (m && PyModule_AddStringConstant(m, "torch_version", MOBA_TORCH_VERSION) != 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
