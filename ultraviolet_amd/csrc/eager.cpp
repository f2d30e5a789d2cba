// decode_attention and varlen_attention (with its gradients) on plain device tensors as one native call each: the checks of the Python path,
// the outputs' allocation, the argument block and the launch.  Whatever is not the plain case comes back as None, and the caller's
// general path takes (or refuses) it.
//
// Why native: 256 rows of up to 1024 keys take the GPU 6.3 us and took the host 11.8 (6.8 a call now, the GPU at work throughout) - 3.3 to fill the argument block field by
// field, 3.2 to launch, 2.0 to allocate the output, the rest to look at shapes and modes.
#include <torch/csrc/python_headers.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
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
// (gradients: whether they may be asked for)
bool plain(PyObject* const* t, int n, bool gradients = false) {
  const uint64_t on = c10::impl::tls_local_dispatch_key_set().included_.raw_repr();
  const c10::DispatchKeySet base(c10::DispatchKey::BackendSelect);
  if (on != base.raw_repr() && on != base.add(c10::DispatchKey::ADInplaceOrView).raw_repr()) return false;
  if (at::impl::PythonTorchFunctionTLS::stack_len() != 0) return false;
  for (int i = 0; i < n; i++) {
    if (t[i] == Py_None && i >= 3) continue;
    if (!is_tensor(t[i]) || (!gradients && THPVariable_Unpack(t[i]).requires_grad())) return false;
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
  const int fp32 = PyObject_IsTrue(args[13]);
  if (fp32 < 0) return nullptr;
  if (!as_int(args[14], a.chunk_keys)) Py_RETURN_NONE;
  at::Tensor out, ws;
  auto allocate = [&] {
    out = at::empty(q.sizes(), fp32 ? q.options().dtype(at::kFloat) : q.options());
    a.out = out.data_ptr(); a.out_dtype = dtype_code(out); a.sob = out.stride(0); a.soh = out.stride(1);
  };
  if (args[12] != Py_None) {
    if (!as_int(args[12], a.num_splits)) Py_RETURN_NONE;
    allocate();
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
    allocate();
    // (how a row is best cut depends on the kernel that serves the call, which its strides and addresses have a say in)
    // (the generic kernel's rule cuts wherever the other one does: where it does not, there is nothing to ask)
    const int64_t work = static_cast<int64_t>(a.B) * a.KH;
    const int generic = uvmi_default_splits(work, ctx, cus);
    a.num_splits = 1;
    if (generic > 1) a.num_splits = uvmi_decode_attn_path(&a) == 1 ? uvmi_decode_attn_splits(qd, kd, work, a.H / a.KH, a.hd, a.S, a.ring, ctx, cus) : generic;
  }
  THPObjectPtr dev(PyLong_FromLong(q.get_device()));
  THPObjectPtr st(dev ? PyObject_CallFunctionObjArgs(raw_stream_fn, dev.get(), nullptr) : nullptr);
  if (!st) return nullptr;
  void* stream = PyLong_AsVoidPtr(st);
  if (PyErr_Occurred()) return nullptr;
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

// ---- varlen_attention: uvmi_prefill_attn and, where a gradient is asked for, a node of the graph whose backward is uvmi_prefill_attn_bwd
struct Packed {   // q, out (1, N, H, 64), k, v (1, N, KH, 64), cu (n_seg + 1)
  uvmi_prefill_attn_args a = {};
  at::Tensor out, ws, lse;
};

// The argument block but for what a call allocates.  False: not the plain case.
bool packed_args(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& cu, double scale, int window, uvmi_prefill_attn_args& a) {
  for (const at::Tensor* t : {&q, &k, &v})
    if (!t->is_cuda() || t->layout() != at::kStrided || t->dim() != 4 || t->size(0) != 1 || t->stride(3) != 1 || t->scalar_type() != q.scalar_type() ||
        t->get_device() != q.get_device() || t->size(1) != q.size(1) || t->size(3) != 64)
      return false;
  if (!cu.is_cuda() || cu.get_device() != q.get_device() || cu.layout() != at::kStrided || cu.dim() != 1 || !cu.is_contiguous()) return false;
  const int dt = dtype_code(q), id = dtype_code(cu);
  if ((dt != UVMI_F16 && dt != UVMI_BF16) || (id != UVMI_I32 && id != UVMI_I64)) return false;
  const int64_t N = q.size(1), H = q.size(2), KH = k.size(2);
  if (N <= 0 || N >= (1 << 30) || KH <= 0 || H > 4096 || H % KH != 0 || v.size(2) != KH || cu.numel() < 2 || cu.numel() > INT_MAX) return false;
  a.q = q.data_ptr(); a.q_dtype = dt; a.sqn = q.stride(1); a.sqh = q.stride(2);
  a.k = k.data_ptr(); a.v = v.data_ptr(); a.kv_dtype = dt;
  a.skn = k.stride(1); a.skh = k.stride(2); a.svn = v.stride(1); a.svh = v.stride(2);
  a.cu_seqlens = cu.data_ptr(); a.idx_dtype = id; a.n_seg = static_cast<int>(cu.numel() - 1);
  a.out_dtype = dt; a.son = H * 64; a.soh = 64;
  a.N = static_cast<int>(N); a.H = static_cast<int>(H); a.KH = static_cast<int>(KH); a.hd = 64;
  a.scale = static_cast<float>(scale); a.window = window;
  return true;
}

// What a call allocates, in the tensors of the Python path.  False: another kernel than the MFMA one would serve it.
bool packed_alloc(const at::Tensor& q, Packed& p, bool statistics) {
  const int64_t N = p.a.N, H = p.a.H;
  p.out = at::empty({1, N, H, 64}, q.options());
  p.a.workspace_bytes = uvmi_prefill_attn_workspace_bytes(p.a.N);
  p.ws = at::empty({static_cast<int64_t>(p.a.workspace_bytes)}, q.options().dtype(at::kByte));
  p.a.out = p.out.data_ptr();
  p.a.workspace = p.ws.data_ptr();
  if (uvmi_prefill_attn_path(&p.a) != 1) return false;
  if (statistics) {   // (varlen_attn.statistics_pitch)
    p.lse = at::empty({H, (N + 31) / 32 * 32 + 32}, q.options().dtype(at::kFloat));
    p.a.lse_out = static_cast<float*>(p.lse.data_ptr());
    p.a.lse_stride = p.lse.stride(0);
  }
  return true;
}

int packed_launch(const Packed& p) { return uvmi_prefill_attn(&p.a, c10::hip::getCurrentHIPStream(p.out.get_device()).stream()); }

// The counterpart of varlen_attn._PackedAttention.  Why it is native: the backward in Python runs on the engine's thread, which has to be handed the
// interpreter first, so the gradients of a few hundred tokens took the host 73 or 137 us, by how the two threads happened to meet; 12 sequences of up
// to 80 tokens, forward and backward, 136 us (73 in its better runs) -> 56, 23 of up to 403 with a window 137 (73) -> 72, of the GPU's time
// now; 31 700 tokens 139 -> 136.
struct PackedAttention : torch::autograd::Function<PackedAttention> {
  static at::Tensor forward(torch::autograd::AutogradContext* ctx, const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& cu,
                            const Packed& p, int* rc) {
    *rc = packed_launch(p);
    ctx->save_for_backward({q, k, v, p.out, cu, p.lse, p.ws});
    ctx->saved_data["scale"] = static_cast<double>(p.a.scale);
    ctx->saved_data["window"] = static_cast<int64_t>(p.a.window);
    return p.out;
  }
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, const torch::autograd::variable_list& grads) {
    const torch::autograd::variable_list s = ctx->get_saved_variables();
    const at::Tensor go = grads[0].contiguous(), q = s[0].contiguous(), k = s[1].contiguous(), v = s[2].contiguous(), o = s[3].contiguous();
    const at::Tensor &cu = s[4], &lse = s[5], &fwd_ws = s[6];
    // (a hook may have put other tensors in the saved ones' place)
    TORCH_CHECK(go.sizes() == q.sizes() && o.sizes() == q.sizes() && k.sizes() == v.sizes() && go.scalar_type() == q.scalar_type() && k.scalar_type() == q.scalar_type() &&
                    v.scalar_type() == q.scalar_type() && o.scalar_type() == q.scalar_type(), "varlen_attention: operands of the backward do not match");
    for (const at::Tensor* t : {&go, &q, &k, &v, &o, &cu, &lse, &fwd_ws}) TORCH_CHECK(t->is_cuda(), "libuvmi kernels need device tensors (there is no CPU path)");
    TORCH_CHECK(cu.is_contiguous() && (cu.scalar_type() == at::kInt || cu.scalar_type() == at::kLong) && lse.dim() == 2 && lse.stride(1) == 1 &&
                    lse.scalar_type() == at::kFloat && fwd_ws.is_contiguous(), "varlen_attention: operands of the backward do not match");
    uvmi_prefill_attn_bwd_args a = {};
    a.N = static_cast<int>(q.size(1)); a.H = static_cast<int>(q.size(2)); a.KH = static_cast<int>(k.size(2)); a.hd = static_cast<int>(q.size(3));
    const at::Tensor dq = at::empty(q.sizes(), q.options()), dk = at::empty(k.sizes(), k.options()), dv = at::empty(v.sizes(), v.options());
    a.workspace_bytes = uvmi_prefill_attn_bwd_workspace_bytes(a.N, a.H);
    const at::Tensor ws = at::empty({static_cast<int64_t>(a.workspace_bytes)}, q.options().dtype(at::kByte));
    a.q = q.data_ptr(); a.k = k.data_ptr(); a.v = v.data_ptr(); a.o = o.data_ptr(); a.go = go.data_ptr(); a.dtype = dtype_code(q);
    a.dq = dq.data_ptr(); a.dk = dk.data_ptr(); a.dv = dv.data_ptr();
    a.cu_seqlens = cu.data_ptr(); a.idx_dtype = dtype_code(cu); a.n_seg = static_cast<int>(cu.numel() - 1);
    a.scale = static_cast<float>(ctx->saved_data["scale"].toDouble()); a.window = static_cast<int>(ctx->saved_data["window"].toInt());
    a.workspace = ws.data_ptr();
    a.lse = static_cast<const float*>(lse.data_ptr()); a.lse_stride = lse.stride(0); a.fwd_workspace = fwd_ws.data_ptr();
    const int rc = uvmi_prefill_attn_bwd(&a, c10::hip::getCurrentHIPStream(q.get_device()).stream());
    TORCH_CHECK(rc == UVMI_OK, "uvmi_prefill_attn_bwd failed (", rc, "): ", uvmi_last_error());
    return {dq, dk, dv, at::Tensor(), at::Tensor(), at::Tensor()};
  }
};

// varlen_attention(q, k, v, cu_seqlens, scale, window) -> as decode_attention above
PyObject* py_varlen_attention(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 6) { PyErr_SetString(PyExc_TypeError, "varlen_attention takes 6 arguments"); return nullptr; }
  touched = 1;
  if (!plain(args, 3, true) || !is_tensor(args[3])) Py_RETURN_NONE;
  const at::Tensor& q = THPVariable_Unpack(args[0]);
  const at::Tensor& k = THPVariable_Unpack(args[1]);
  const at::Tensor& v = THPVariable_Unpack(args[2]);
  const at::Tensor& cu = THPVariable_Unpack(args[3]);
  int window = 0;
  if (!PyFloat_Check(args[4]) || (args[5] != Py_None && !as_int(args[5], window))) Py_RETURN_NONE;
  Packed p;
  if (!packed_args(q, k, v, cu, PyFloat_AS_DOUBLE(args[4]), window, p.a)) Py_RETURN_NONE;
  const bool graph = at::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad());
  if (!packed_alloc(q, p, graph)) Py_RETURN_NONE;
  int rc = UVMI_OK;
  at::Tensor out = p.out;
  if (graph) out = PackedAttention::apply(q, k, v, cu, p, &rc);
  else rc = packed_launch(p);
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
    {"varlen_attention", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_varlen_attention)), METH_FASTCALL, nullptr},
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
      PyModule_AddIntConstant(m.get(), "attn_args_bytes", sizeof(uvmi_attn_args)) ||
      PyModule_AddIntConstant(m.get(), "prefill_attn_args_bytes", sizeof(uvmi_prefill_attn_args)) ||
      PyModule_AddIntConstant(m.get(), "prefill_attn_bwd_args_bytes", sizeof(uvmi_prefill_attn_bwd_args)))
    return nullptr;
  return m.release();
}
