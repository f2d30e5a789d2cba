// decode_attention on plain device tensors as one native call: the checks of the Python path, the output's allocation, the argument
// block and the launch.  Whatever is not the plain case comes back as None, and the caller's general path takes (or refuses) it.
//
// Why native: 256 rows of up to 1024 keys take the GPU 6.3 us and took the host 11.8 (6.8 a call now, the GPU at work throughout) - 3.3 to fill the argument block field by
// field, 3.2 to launch, 2.0 to allocate the output, the rest to look at shapes and modes.
#include <torch/csrc/python_headers.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>

#include <atomic>
#include <climits>

#include "../../include/uvmi.h"

namespace {

PyObject* raw_stream_fn = nullptr;   // torch._C._cuda_getCurrentRawStream
PyObject* device_cus_fn = nullptr;   // decode_attn._device_cus, set once by bind()
std::atomic<int> device_cus[64];
// Accessed in every call: this module is loaded behind the others, and until a thread has accessed a thread-local of it, glibc before 2.39 sends
// every access to theirs the slow way (6 rows sampled from Python after a call of this module 9.0 us, 7.6 so; the call itself 5.1, 4.4)
thread_local volatile char touched;

bool is_tensor(PyObject* o) { return Py_TYPE(o) == reinterpret_cast<PyTypeObject*>(THPVariableClass); }

int dtype_code(const at::Tensor& t) {
  switch (t.scalar_type()) {
    case at::kHalf: return UVMI_F16;
    case at::kBFloat16: return UVMI_BF16;
    case at::kFloat: return UVMI_F32;
    case at::kChar: return UVMI_I8;
    case at::kInt: return UVMI_I32;
    case at::kLong: return UVMI_I64;
    default: return -1;
  }
}

// decode_attn.plain_eager but for the two questions that only Python answers (compiling, forward-mode level)
bool plain(PyObject* const* t, int n) {
  const uint64_t on = c10::impl::tls_local_dispatch_key_set().included_.raw_repr();
  const c10::DispatchKeySet base(c10::DispatchKey::BackendSelect);
  if (on != base.raw_repr() && on != base.add(c10::DispatchKey::ADInplaceOrView).raw_repr()) return false;
  if (at::impl::PythonTorchFunctionTLS::stack_len() != 0) return false;
  for (int i = 0; i < n; i++) {
    if (t[i] == Py_None && i >= 3) continue;
    if (!is_tensor(t[i]) || THPVariable_Unpack(t[i]).requires_grad()) return false;
  }
  return true;
}

bool as_int(PyObject* o, int& v) {
  if (!PyLong_Check(o)) return false;
  int over = 0;
  const long x = PyLong_AsLongAndOverflow(o, &over);
  if (over || x < INT_MIN || x > INT_MAX) return false;
  v = static_cast<int>(x);
  return true;
}

// plain(q, k, v, k_scale, v_scale)
PyObject* py_plain(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 5) { PyErr_SetString(PyExc_TypeError, "plain takes 5 arguments"); return nullptr; }
  return PyBool_FromLong(plain(args, 5));
  END_HANDLE_TH_ERRORS
}

// decode_attention(q, k_cache, v_cache, k_scale, v_scale, pos, starts, rows, scale, window, ring, ctx_hint, num_splits, out_fp32, chunk_keys)
// -> the output; None where the call is not plain; an int, the library's error code, where it was refused
PyObject* py_decode_attention(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 15) { PyErr_SetString(PyExc_TypeError, "decode_attention takes 15 arguments"); return nullptr; }
  touched = 1;
  if (!plain(args, 5)) Py_RETURN_NONE;
  const at::Tensor& q = THPVariable_Unpack(args[0]);
  const at::Tensor& k = THPVariable_Unpack(args[1]);
  const at::Tensor& v = THPVariable_Unpack(args[2]);
  if (!is_tensor(args[5]) || !is_tensor(args[6]) || (args[7] != Py_None && !is_tensor(args[7]))) Py_RETURN_NONE;
  const at::Tensor& pos = THPVariable_Unpack(args[5]);
  const at::Tensor& starts = THPVariable_Unpack(args[6]);
  if (!q.is_cuda() || !k.is_cuda() || !v.is_cuda() || !pos.is_cuda() || !starts.is_cuda()) Py_RETURN_NONE;
  if (q.layout() != at::kStrided || k.layout() != at::kStrided || v.layout() != at::kStrided) Py_RETURN_NONE;
  if (q.dim() != 3 || k.dim() != 4 || v.dim() != 4 || q.stride(2) != 1 || k.stride(3) != 1 || v.stride(3) != 1) Py_RETURN_NONE;
  const int qd = dtype_code(q), kd = dtype_code(k), id = dtype_code(pos);
  if (qd < 0 || kd < 0 || (id != UVMI_I32 && id != UVMI_I64) || starts.scalar_type() != pos.scalar_type()) Py_RETURN_NONE;
  if (!pos.is_contiguous() || !starts.is_contiguous()) Py_RETURN_NONE;
  if (q.size(0) > INT_MAX || q.size(1) > INT_MAX || q.size(2) > INT_MAX || k.size(1) > INT_MAX || k.size(2) > INT_MAX) Py_RETURN_NONE;
  uvmi_attn_args a = {};
  a.q = q.data_ptr(); a.q_dtype = qd; a.sqb = q.stride(0); a.sqh = q.stride(1);
  a.k_cache = k.data_ptr(); a.v_cache = v.data_ptr(); a.kv_dtype = kd;
  a.skb = k.stride(0); a.skh = k.stride(1); a.sks = k.stride(2);
  a.svb = v.stride(0); a.svh = v.stride(1); a.svs = v.stride(2);
  if (kd == UVMI_I8) {
    if (args[3] == Py_None || args[4] == Py_None) Py_RETURN_NONE;
    const at::Tensor& ks = THPVariable_Unpack(args[3]);
    const at::Tensor& vs = THPVariable_Unpack(args[4]);
    if (ks.dim() != 3 || vs.dim() != 3 || ks.stride(2) != 1 || vs.stride(2) != 1) Py_RETURN_NONE;
    a.k_scale = ks.data_ptr(); a.v_scale = vs.data_ptr();
    a.ssb = ks.stride(0); a.ssh = ks.stride(1); a.stb = vs.stride(0); a.sth = vs.stride(1);
  }
  a.pos = pos.data_ptr(); a.starts = starts.data_ptr(); a.idx_dtype = id;
  a.B = static_cast<int>(q.size(0)); a.H = static_cast<int>(q.size(1)); a.hd = static_cast<int>(q.size(2));
  a.KH = static_cast<int>(k.size(1)); a.S = static_cast<int>(k.size(2));
  if (args[7] != Py_None) {
    const at::Tensor& rows = THPVariable_Unpack(args[7]);
    if (!rows.is_cuda() || rows.scalar_type() != pos.scalar_type() || !rows.is_contiguous() || rows.numel() != a.B) Py_RETURN_NONE;
    a.rows = rows.data_ptr();
  }
  if (PyFloat_Check(args[8])) a.scale = static_cast<float>(PyFloat_AS_DOUBLE(args[8]));
  else Py_RETURN_NONE;
  if (!as_int(args[9], a.window)) Py_RETURN_NONE;
  if (args[10] == Py_None) a.ring = a.window > 0;
  else if (PyBool_Check(args[10])) a.ring = args[10] == Py_True;
  else Py_RETURN_NONE;
  if (args[12] != Py_None) {
    if (!as_int(args[12], a.num_splits)) Py_RETURN_NONE;
  } else {
    int ctx = 0;
    if (args[11] != Py_None && !as_int(args[11], ctx)) Py_RETURN_NONE;
    if (ctx == 0) ctx = a.S;
    if (a.window > 0 && a.window < ctx) ctx = a.window;
    const int dev = q.get_device();
    if (dev >= 64 || ctx < 0) Py_RETURN_NONE;
    int cus = device_cus[dev].load(std::memory_order_relaxed);
    if (cus == 0) {
      THPObjectPtr idx(PyLong_FromLong(dev));
      THPObjectPtr r(idx ? PyObject_CallFunctionObjArgs(device_cus_fn, idx.get(), nullptr) : nullptr);
      if (!r || !as_int(r, cus)) return nullptr;
      device_cus[dev].store(cus, std::memory_order_relaxed);
    }
    a.num_splits = uvmi_decode_attn_splits(qd, kd, static_cast<int64_t>(a.B) * a.KH, a.KH > 0 ? a.H / a.KH : 0, a.hd, a.S, a.ring, ctx, cus);
  }
  const int fp32 = PyObject_IsTrue(args[13]);
  if (fp32 < 0) return nullptr;
  if (!as_int(args[14], a.chunk_keys)) Py_RETURN_NONE;
  THPObjectPtr dev(PyLong_FromLong(q.get_device()));
  THPObjectPtr st(dev ? PyObject_CallFunctionObjArgs(raw_stream_fn, dev.get(), nullptr) : nullptr);
  if (!st) return nullptr;
  void* stream = PyLong_AsVoidPtr(st);
  if (PyErr_Occurred()) return nullptr;
  at::Tensor out = at::empty(q.sizes(), fp32 ? q.options().dtype(at::kFloat) : q.options()), ws;
  a.out = out.data_ptr(); a.out_dtype = dtype_code(out); a.sob = out.stride(0); a.soh = out.stride(1);
  if (a.num_splits > 1) {
    a.workspace_bytes = uvmi_decode_attn_workspace_bytes(a.B, a.H, a.KH, a.hd, a.num_splits);
    ws = at::empty({static_cast<int64_t>(a.workspace_bytes)}, q.options().dtype(at::kByte));
    a.workspace = ws.data_ptr();
  }
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = uvmi_decode_attn(&a, stream);
  Py_END_ALLOW_THREADS
  if (rc != UVMI_OK) return PyLong_FromLong(rc);
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// bind(device_cus): the function that answers how many compute units a device has
PyObject* py_bind(PyObject*, PyObject* fn) {
  Py_INCREF(fn);
  Py_XSETREF(device_cus_fn, fn);
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"plain", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_plain)), METH_FASTCALL, nullptr},
    {"decode_attention", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_decode_attention)), METH_FASTCALL, nullptr},
    {"bind", py_bind, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "uvmi_eager", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_uvmi_eager() {
  THPObjectPtr c(PyImport_ImportModule("torch._C"));
  if (!c) return nullptr;
  raw_stream_fn = PyObject_GetAttrString(c, "_cuda_getCurrentRawStream");
  if (!raw_stream_fn) return nullptr;
  THPObjectPtr m(PyModule_Create(&module));
  // what the loader compares with its own: the revision and layout this was built for, and the revision of the library it calls
  if (!m || PyModule_AddIntConstant(m.get(), "revision", UVMI_ABI_VERSION) || PyModule_AddIntConstant(m.get(), "library_revision", uvmi_version()) ||
      PyModule_AddIntConstant(m.get(), "attn_args_bytes", sizeof(uvmi_attn_args)))
    return nullptr;
  return m.release();
}
