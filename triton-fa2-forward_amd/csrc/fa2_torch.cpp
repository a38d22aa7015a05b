// fa2_torch.cpp - fa2/_torch_call.so: the common call of fa2.kernel.attention, made natively.
//
// attention()'s checks, policy, allocations and launch took 11-17 us per call in Python and ctypes
// (a causal call of B1 H4 N256 D64 11.2 us, a split-KV one 16.5), more than the kernels of a short
// prompt or a decoding step run for (5-10 us), so back-to-back calls waited for the host. Here the
// same steps on at::Tensor take about 4 us, the launch included.
//
// call() takes exactly the calls that need nothing else: plain dense GPU tensors of the current
// device that satisfy every check of attention() and the library's 16-byte rule, with default
// tiles, packing and split count. Anything else returns None, and attention()'s Python does it: it
// raises the reference's errors, copies tensors the kernel cannot load, switches devices, honours
// the overrides. No state is kept from one call to the next.
#include <Python.h>

#include <ATen/TensorSubclassLikeUtils.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/empty_like.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/PythonTorchFunctionTLS.h>

#include <atomic>
#include <climits>
#include <cmath>
#include <cstdint>

#include "fa2_fwd.h"

namespace {

constexpr double kLog2e = 1.4426950408889634;       // fa2/kernel.py: LOG2E
constexpr int64_t kMaxKvRowStride = int64_t(1) << 22;  // fa2/kernel.py: _MAX_KV_ROW_STRIDE
constexpr int kMaxDevices = 64;

// The device's CU count, as torch.cuda.get_device_properties reports it; 0 if unknown.
int cu_count(int dev) {
  static std::atomic<int> cus[kMaxDevices];
  if (dev < 0 || dev >= kMaxDevices) return 0;
  int n = cus[dev].load(std::memory_order_relaxed);
  if (n == 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) {
      (void)hipGetLastError();
      return 0;
    }
    cus[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}

// A tensor whose memory the kernel may address through data_ptr: no subclass, no wrapper of a
// transform, strided and on the GPU.
bool plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return false;
  const at::Tensor& t = THPVariable_Unpack(o);
  return t.defined() && t.dim() == 4 && t.layout() == at::kStrided && t.is_cuda() &&
         t.has_storage() && !t.is_conj() && !t.is_neg() && !at::isTensorSubclassLike(t);
}

// The element strides the library takes (0 for a dimension of one element, which it never steps),
// and whether its 16-byte loads can address the tensor: fa2/kernel.py's _loadable.
bool strides_of(const at::Tensor& t, int64_t max_row, int64_t (&s)[4]) {
  if (reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 || t.stride(3) != 1) return false;
  for (int i = 0; i < 3; ++i) {
    s[i] = t.size(i) == 1 ? 0 : t.stride(i);
    if (s[i] % 8) return false;
  }
  s[3] = 1;
  return s[2] <= max_row;
}

// attention()'s policy at the default tiles: packing, split count and workspace. The count is the one
// that runs, which needs the smaller workspace, unless the workspace has room for the key-norm table:
// the kernel that uses the table takes fa2_num_splits's count, as fa2_launch_splits's contract says.
struct Policy {
  int32_t bm = 0, bn = 0, pack = 1, splits = 1;
  size_t ws_bytes = 0;
};
bool policy_of(int32_t B, int32_t hq, int32_t hkv, int32_t nq, int32_t nkv, int32_t D, int32_t dtype,
               int32_t causal, int32_t cus, Policy* out) {
  Policy p;
  if (fa2_default_config(D, &p.bm, &p.bn, nullptr, nullptr) != FA2_OK) return false;
  if (fa2_should_pack_gqa(nq, hq / hkv, p.bm)) p.pack = hq / hkv;
  if (!causal) p.splits = fa2_num_splits(B, hq, hkv, nq, nkv, D, 0, p.bm, p.bn, cus);
  p.ws_bytes = fa2_workspace_bytes_for(B, hq, hkv, nq, nkv, D, dtype, causal, p.splits);
  if (p.splits > 1 && p.ws_bytes == fa2_workspace_bytes(B, hq, nq, D, p.splits)) {
    p.splits = fa2_launch_splits(B, hq, hkv, nq, nkv, D, 0, p.bm, p.bn, cus, p.splits);
    p.ws_bytes = fa2_workspace_bytes(B, hq, nq, D, p.splits);
  }
  *out = p;
  return true;
}

// policy(batch, h_q, h_kv, n_q, n_kv, head_dim, dtype, causal, cus) -> (pack, splits, workspace bytes)
// of a call of these sizes on a GPU of `cus` CUs (dtype: the C ABI's code). No GPU call.
PyObject* policy(PyObject*, PyObject* args) {
  int B, hq, hkv, nq, nkv, D, dtype, causal, cus;
  if (!PyArg_ParseTuple(args, "iiiiiiiii", &B, &hq, &hkv, &nq, &nkv, &D, &dtype, &causal, &cus))
    return nullptr;
  Policy p;
  if (B < 1 || hkv < 1 || hq < 1 || hq % hkv || nq < 1 || nkv < 1 || cus < 1 ||
      !policy_of(B, hq, hkv, nq, nkv, D, dtype, causal, cus, &p)) {
    PyErr_SetString(PyExc_ValueError, "sizes that attention() rejects");
    return nullptr;
  }
  return Py_BuildValue("iin", p.pack, p.splits, (Py_ssize_t)p.ws_bytes);
}

// call(q, k, v, causal, sm_scale, return_lse) -> attention()'s result, or None (see above)
PyObject* call(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  if (n_args != 6) {
    PyErr_SetString(PyExc_TypeError, "call(q, k, v, causal, sm_scale, return_lse)");
    return nullptr;
  }
  if (!plain(args[0]) || !plain(args[1]) || !plain(args[2]) ||
      c10::impl::dispatch_mode_enabled() || at::impl::torch_function_mode_enabled())
    Py_RETURN_NONE;
  const at::Tensor& q = THPVariable_Unpack(args[0]);
  const at::Tensor& k = THPVariable_Unpack(args[1]);
  const at::Tensor& v = THPVariable_Unpack(args[2]);
  const int causal = PyObject_IsTrue(args[3]);
  const int want_lse = PyObject_IsTrue(args[5]);
  if (causal < 0 || want_lse < 0) return nullptr;

  // ---- attention()'s checks (fa2/kernel.py:218-228 of the reference)
  const int64_t B = q.size(0), hq = q.size(1), nq = q.size(2), D = q.size(3);
  const int64_t hkv = k.size(1), nkv = k.size(2);
  const auto dtype = q.scalar_type();
  if ((dtype != at::kHalf && dtype != at::kBFloat16) || k.scalar_type() != dtype ||
      v.scalar_type() != dtype || k.sizes() != v.sizes() || k.size(0) != B || k.size(3) != D ||
      (D != 16 && D != 32 && D != 64 && D != 128))
    Py_RETURN_NONE;
  if (B < 1 || hkv < 1 || hq < 1 || nq < 1 || nkv < 1 || hq % hkv || (causal && nq != nkv) ||
      B > INT32_MAX || hq > INT32_MAX || nq > INT32_MAX || nkv > INT32_MAX)
    Py_RETURN_NONE;
  const auto device = q.device();
  if (k.device() != device || v.device() != device || device.index() != c10::hip::current_device())
    Py_RETURN_NONE;
  double sm_scale = 1.0 / std::sqrt((double)D);
  if (args[4] != Py_None) {
    if (!PyFloat_CheckExact(args[4])) Py_RETURN_NONE;
    sm_scale = PyFloat_AS_DOUBLE(args[4]);
    if (!(sm_scale > 0)) Py_RETURN_NONE;
  }
  int64_t sq[4], sk[4], sv[4], so[4];
  if (!strides_of(q, INT64_MAX, sq) || !strides_of(k, kMaxKvRowStride, sk) ||
      !strides_of(v, kMaxKvRowStride, sv))
    Py_RETURN_NONE;

  const int cus = causal ? 1 : cu_count(device.index());
  const int32_t code = dtype == at::kBFloat16 ? FA2_DTYPE_BF16 : FA2_DTYPE_F16;
  Policy p;
  if (cus < 1 || nq > INT32_MAX / (hq / hkv) ||
      !policy_of((int32_t)B, (int32_t)hq, (int32_t)hkv, (int32_t)nq, (int32_t)nkv, (int32_t)D, code,
                 causal, cus, &p))
    Py_RETURN_NONE;

  // ---- outputs, workspace, launch
  at::Tensor out = at::empty_like(q);
  if (!strides_of(out, INT64_MAX, so)) Py_RETURN_NONE;
  at::Tensor lse, ws;
  if (want_lse) lse = at::empty({B, hq, nq}, q.options().dtype(at::kFloat));
  if (p.ws_bytes) ws = at::empty({(int64_t)p.ws_bytes}, q.options().dtype(at::kByte));
  void* stream = c10::hip::getCurrentHIPStream(device.index()).stream();
  const void *qp = q.data_ptr(), *kp = k.data_ptr(), *vp = v.data_ptr();
  void* op = out.data_ptr();
  float* lp = want_lse ? static_cast<float*>(lse.data_ptr()) : nullptr;
  void* wp = p.ws_bytes ? ws.data_ptr() : nullptr;
  int rc;
  Py_BEGIN_ALLOW_THREADS  // as ctypes does around a foreign call
  rc = fa2_attn_fwd_ex(qp, kp, vp, op, sq, sk, sv, so, (int32_t)B, (int32_t)hq, (int32_t)hkv,
                       (int32_t)nq, (int32_t)nkv, (int32_t)D, code, causal, p.pack, p.bm, p.bn,
                       (float)(sm_scale * kLog2e), lp, p.splits, wp, p.ws_bytes, stream);
  Py_END_ALLOW_THREADS
  if (rc != FA2_OK) Py_RETURN_NONE;  // nothing ran: attention() repeats the call and raises
  PyObject* o = THPVariable_Wrap(std::move(out));
  if (!o || !want_lse) return o;
  PyObject* l = THPVariable_Wrap(std::move(lse));
  if (!l) {
    Py_DECREF(o);
    return nullptr;
  }
  PyObject* both = PyTuple_Pack(2, o, l);
  Py_DECREF(o);
  Py_DECREF(l);
  return both;
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"call", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(call)), METH_FASTCALL,
     "call(q, k, v, causal, sm_scale, return_lse) -> attention()'s result, or None"},
    {"policy", policy, METH_VARARGS,
     "policy(batch, h_q, h_kv, n_q, n_kv, head_dim, dtype, causal, cus) -> (pack, splits, workspace bytes)"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_torch_call", nullptr, -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

// built_for: fa2/_lib.py's build_id() of the torch and Python compiled against (csrc/build.py); another
// one does not use this module.
PyMODINIT_FUNC PyInit__torch_call() {
  PyObject* m = PyModule_Create(&module);
  if (m && PyModule_AddStringConstant(m, "built_for", FA2_BUILT_FOR) < 0) Py_CLEAR(m);
  return m;
}
