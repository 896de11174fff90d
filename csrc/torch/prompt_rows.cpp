// The operators of a prompt's layer (LayerNorm of rows, products of few rows, rotation into the cache, packed attention) without Python
// frames: argument checks, allocations and the launch in C++. Each returns None for a call that the same function in Python
// (ops/norms.py, ops/linear.py, ops/rope.py, ops/attention.py) is to take: gradients, transforms, modes, traces, autocast, tensors of other
// types or places.
//
// Why: a prompt of few rows is bound by the host. 61 tokens through four GPT-J layers of 4096 are 460 us of kernels that took 560 us to
// issue, 11 to 22 us a launch, mostly checks and ctypes' conversions; so 375.
#include "prompt_rows.h"

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/autocast_mode.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/csrc/utils/object_ptr.h>

namespace {

using at::Tensor;
typedef long long ll;

// of the kernel library that ops/_lib.py has loaded
typedef int (*RowsFn)(int, int, const void*, const void*, const void*, void*, int, int, int, const void*, const void*, const void*, void*,
                      int, int, int, const void*, float*, unsigned*, ll, int, int, int, hipStream_t);
typedef int (*NormFn)(const void*, const void*, const void*, void*, const void*, const void*, void*, float*, float*, int, int, float,
                      hipStream_t);
typedef int (*NormF16Fn)(const void*, ll, const void*, const void*, void*, ll, const void*, const void*, float, void*, int, int,
                         hipStream_t);
typedef int (*AppendFn)(int, void*, void*, const void*, ll, ll, ll, ll, ll, ll, int, int, int, int, int, int, const float*, const float*,
                        const int*, const int*, const int*, void*, void*, int, hipStream_t);
typedef int (*PackedFn)(int, const void*, const void*, const void*, void*, ll, ll, ll, ll, ll, ll, ll, ll, int, int, int, int, int, int,
                        float, const float*, int, const int*, int*, hipStream_t);
RowsFn rows_mm = nullptr;
NormFn norm = nullptr;
NormF16Fn norm_f16 = nullptr;
AppendFn append = nullptr;
PackedFn packed = nullptr;
PyObject* counters = nullptr;  // ops/_lib.py's, of the current stream

// An eager call without gradients, transforms, modes, tracing or autocast
bool plain_inference() {
  return !c10::GradMode::is_enabled() && !at::autocast::is_autocast_enabled(at::kCUDA) &&
         !c10::impl::TorchDispatchModeTLS::any_modes_set() && !at::impl::torch_function_mode_enabled() &&
         !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) && !torch::jit::tracer::isTracing();
}
bool is_tensor(PyObject* o) { return THPVariable_CheckExact(o); }
bool is_tensor_or_none(PyObject* o) { return o == Py_None || THPVariable_CheckExact(o); }
bool on(const Tensor& t, int64_t device) {
  return t.is_cuda() && t.get_device() == device && t.layout() == at::kStrided && !t._fw_grad(0).defined();
}
const void* at_or_null(PyObject* o) { return o == Py_None ? nullptr : THPVariable_Unpack(o).const_data_ptr(); }
bool aligned(const Tensor& t) { return reinterpret_cast<uintptr_t>(t.const_data_ptr()) % 16 == 0; }
hipStream_t stream_of(int64_t device) { return c10::hip::getCurrentHIPStream(device).stream(); }
bool half_type(const Tensor& t) { return t.scalar_type() == at::kBFloat16 || t.scalar_type() == at::kHalf; }

bool bias_fits(PyObject* o, int64_t n, const Tensor& x, int64_t device) {
  if (o == Py_None) return true;
  const Tensor& b = THPVariable_Unpack(o);
  return on(b, device) && b.dim() == 1 && b.size(0) == n && b.scalar_type() == x.scalar_type() && b.is_contiguous();
}

}  // namespace

// few_rows(x, weight, bias | None, x2 | None, weight2, bias2 | None, act, act2, beside, rows[, res | None]) -> (y,) or (y, y2), or None. The
// caller has asked few_rows (ops/linear.py) about the sizes.
PyObject* kca_few_rows(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if ((n != 10 && n != 11) || !rows_mm) {
    PyErr_SetString(PyExc_TypeError, "few_rows(x, weight, bias, x2, weight2, bias2, act, act2, beside, rows, res) after init_rows");
    return nullptr;
  }
  const int parts = a[3] == Py_None ? 1 : 2;
  PyObject* const res = n > 10 ? a[10] : Py_None;
  for (int i = 0; i < parts; ++i)
    if (!is_tensor(a[3 * i]) || !is_tensor(a[3 * i + 1]) || !is_tensor_or_none(a[3 * i + 2])) Py_RETURN_NONE;
  if (!is_tensor_or_none(res)) Py_RETURN_NONE;
  const long act = PyLong_AsLong(a[6]), act2 = PyLong_AsLong(a[7]), rows = PyLong_AsLong(a[9]);
  const int beside = PyObject_IsTrue(a[8]);
  if (PyErr_Occurred()) return nullptr;
  if (!plain_inference()) Py_RETURN_NONE;
  const Tensor& x0 = THPVariable_Unpack(a[0]);
  if (!x0.is_cuda() || !half_type(x0) || rows < 1 || rows > 128) Py_RETURN_NONE;
  const int64_t device = x0.get_device();
  if (device != c10::hip::current_device() || c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None)
    Py_RETURN_NONE;
  for (int i = 0; i < parts; ++i) {
    const Tensor &x = THPVariable_Unpack(a[3 * i]), &w = THPVariable_Unpack(a[3 * i + 1]);
    if (!on(x, device) || !on(w, device) || w.dim() != 2 || x.scalar_type() != x0.scalar_type() || w.scalar_type() != x0.scalar_type())
      Py_RETURN_NONE;
    const int64_t N = w.size(0), K = w.size(1);
    if (N < 16 || N % 16 || K < 64 || K % 64 || x.numel() != rows * K || !x.is_contiguous() || !w.is_contiguous() || !aligned(x) ||
        !aligned(w) || 2 * std::max<int64_t>(N, rows) * K >= 1ll << 32 || !bias_fits(a[3 * i + 2], N, x, device))
      Py_RETURN_NONE;
  }
  const Tensor &w = THPVariable_Unpack(a[1]), &w2 = THPVariable_Unpack(a[parts > 1 ? 4 : 1]);
  const int64_t N = w.size(0), K = w.size(1), N2 = w2.size(0), K2 = w2.size(1);
  const bool two = parts > 1, apart = two && beside;
  if (two && !beside && N != N2) Py_RETURN_NONE;
  if (res != Py_None) {
    const Tensor& r = THPVariable_Unpack(res);
    if (!two || beside || !on(r, device) || r.scalar_type() != x0.scalar_type() || r.numel() != rows * N || !r.is_contiguous() ||
        reinterpret_cast<uintptr_t>(r.const_data_ptr()) % 8)
      Py_RETURN_NONE;
  }
  // (as _few_launch: about one block of 64 weight rows a CU)
  const int64_t blocks = (N + 63) / 64 + (apart ? (N2 + 63) / 64 : 0), k = apart ? std::min(K, K2) : two ? K + K2 : K;
  const int64_t ks = std::max<int64_t>(1, std::min(256 / blocks, k / 512));
  Tensor y = at::empty({rows, N}, x0.options()), y2, ws, cnt;
  if (apart) y2 = at::empty({rows, N2}, x0.options());
  if (ks > 1) {
    ws = at::empty({blocks * ks * 64 * (rows <= 32 ? 32 : rows <= 64 ? 64 : 128)}, x0.options().dtype(at::kFloat));
    THPObjectPtr dev(PyObject_GetAttrString(a[0], "device")), c(dev ? PyObject_CallFunction(counters, "OL", dev.get(), (ll)blocks) : nullptr);
    if (!c) return nullptr;
    cnt = THPVariable_Unpack(c.get());
  }
  const int rc = rows_mm(x0.scalar_type() == at::kBFloat16 ? 1 : 2, apart, x0.const_data_ptr(), w.const_data_ptr(), at_or_null(a[2]),
                         y.mutable_data_ptr(), N, K, act, two ? at_or_null(a[3]) : nullptr, two ? w2.const_data_ptr() : nullptr,
                         two ? at_or_null(a[5]) : nullptr, apart ? y2.mutable_data_ptr() : nullptr, two ? N2 : 0, two ? K2 : 0,
                         two ? act2 : 0, at_or_null(res), ks > 1 ? ws.mutable_data_ptr<float>() : nullptr,
                         ks > 1 ? reinterpret_cast<unsigned*>(cnt.mutable_data_ptr<int>()) : nullptr, ks > 1 ? ws.numel() : 0,
                         ks > 1 ? cnt.numel() : 0, rows, ks, stream_of(device));
  TORCH_CHECK(rc == 0, "kca_rows_mm_two returned status ", rc, " (unsupported shape/arguments)");
  THPObjectPtr py(THPVariable_Wrap(std::move(y)));
  if (!apart) return PyTuple_Pack(1, py.get());
  THPObjectPtr py2(THPVariable_Wrap(std::move(y2)));
  return PyTuple_Pack(2, py.get(), py2.get());
  END_HANDLE_TH_ERRORS
}

// norm_rows(x, weight, bias | None, eps, r1 | None, r2 | None) -> (y, h) with residuals, else y; or None
PyObject* kca_norm_rows(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 6 || !norm) {
    PyErr_SetString(PyExc_TypeError, "norm_rows(x, weight, bias, eps, r1, r2) after init_rows");
    return nullptr;
  }
  if (c10::GradMode::is_enabled() || !is_tensor(a[0]) || !is_tensor(a[1])) Py_RETURN_NONE;
  for (int i : {2, 4, 5})
    if (!is_tensor_or_none(a[i])) Py_RETURN_NONE;
  const double eps = PyFloat_AsDouble(a[3]);
  if (PyErr_Occurred()) return nullptr;
  if (!plain_inference()) Py_RETURN_NONE;
  const Tensor &x = THPVariable_Unpack(a[0]), &w = THPVariable_Unpack(a[1]);
  if (!x.is_cuda() || !half_type(x) || x.dim() < 1 || x.numel() == 0) Py_RETURN_NONE;
  const int64_t device = x.get_device(), d = x.size(-1), rows = x.numel() / d;
  const bool f16 = x.scalar_type() == at::kHalf;
  if (device != c10::hip::current_device() || d % 8 || d > 16384 || rows >= 1ll << 31 || !on(x, device) || !x.is_contiguous() ||
      !aligned(x) || !on(w, device) || w.dim() != 1 || w.size(0) != d || w.scalar_type() != x.scalar_type() || !w.is_contiguous() ||
      !aligned(w) || !bias_fits(a[2], d, x, device) || (a[2] != Py_None && !aligned(THPVariable_Unpack(a[2]))) ||
      (a[4] == Py_None && a[5] != Py_None))
    Py_RETURN_NONE;
  for (int i : {4, 5}) {
    if (a[i] == Py_None) continue;
    const Tensor& r = THPVariable_Unpack(a[i]);
    if (!on(r, device) || r.scalar_type() != x.scalar_type() || r.sizes() != x.sizes() || !r.is_contiguous() || !aligned(r)) Py_RETURN_NONE;
  }
  const bool sum = a[4] != Py_None;
  Tensor y = at::empty(x.sizes(), x.options()), h;
  if (sum) h = at::empty(x.sizes(), x.options());
  void* hp = sum ? h.mutable_data_ptr() : nullptr;
  const int rc = f16 ? norm_f16(x.const_data_ptr(), d, at_or_null(a[4]), at_or_null(a[5]), hp, d, w.const_data_ptr(), at_or_null(a[2]),
                                (float)eps, y.mutable_data_ptr(), rows, d, stream_of(device))
                     : norm(x.const_data_ptr(), at_or_null(a[4]), at_or_null(a[5]), hp, w.const_data_ptr(), at_or_null(a[2]),
                            y.mutable_data_ptr(), nullptr, nullptr, rows, d, (float)eps, stream_of(device));
  TORCH_CHECK(rc == 0, f16 ? "kca_ln_rows_f16" : "kca_layernorm_fwd", " returned status ", rc, " (unsupported shape/arguments)");
  if (!sum) return THPVariable_Wrap(std::move(y));
  THPObjectPtr py(THPVariable_Wrap(std::move(y))), ph(THPVariable_Wrap(std::move(h)));
  return PyTuple_Pack(2, py.get(), ph.get());
  END_HANDLE_TH_ERRORS
}

namespace {
// rows [T, H, D] of a fused projection
bool prompt_rows(const Tensor& t, const Tensor& q, int64_t device) {
  return on(t, device) && t.dim() == 3 && t.scalar_type() == q.scalar_type() && t.stride(2) == 1 && t.size(0) == q.size(0) &&
         t.size(2) == q.size(2);
}
bool ints(const Tensor& t, int64_t n, int64_t device) {
  return on(t, device) && t.scalar_type() == at::kInt && t.dim() == 1 && t.size(0) == n && t.is_contiguous();
}
bool table(PyObject* o, int64_t device) {
  if (o == Py_None) return true;
  const Tensor& t = THPVariable_Unpack(o);
  return on(t, device) && t.scalar_type() == at::kFloat && t.is_contiguous();
}
}  // namespace

// rope_append(q, k, v, rot, interleaved, cos | None, sin | None, pos, page, off, kc, vc) -> whether the kernel took it, or None
PyObject* kca_rope_rows(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 12 || !append) {
    PyErr_SetString(PyExc_TypeError, "rope_append(q, k, v, rot, interleaved, cos, sin, pos, page, off, kc, vc) after init_rows");
    return nullptr;
  }
  for (int i : {0, 1, 2, 7, 8, 9, 10, 11})
    if (!is_tensor(a[i])) Py_RETURN_NONE;
  if (!is_tensor_or_none(a[5]) || !is_tensor_or_none(a[6])) Py_RETURN_NONE;
  const long rot = PyLong_AsLong(a[3]);
  const int inter = PyObject_IsTrue(a[4]);
  if (PyErr_Occurred()) return nullptr;
  if (!plain_inference()) Py_RETURN_NONE;
  const Tensor &q = THPVariable_Unpack(a[0]), &k = THPVariable_Unpack(a[1]), &v = THPVariable_Unpack(a[2]),
               &kc = THPVariable_Unpack(a[10]), &vc = THPVariable_Unpack(a[11]);
  if (!q.is_cuda() || !half_type(q) || q.dim() != 3) Py_RETURN_NONE;
  const int64_t device = q.get_device(), T = q.size(0);
  if (device != c10::hip::current_device() || !prompt_rows(q, q, device) || !prompt_rows(k, q, device) || !prompt_rows(v, q, device) ||
      k.size(1) != v.size(1) || !on(kc, device) || !on(vc, device) || kc.dim() != 4 || kc.sizes() != vc.sizes() ||
      kc.scalar_type() != q.scalar_type() || vc.scalar_type() != q.scalar_type() || !kc.is_contiguous() || !vc.is_contiguous() ||
      kc.size(1) != k.size(1) || kc.size(3) != q.size(2) || !table(a[5], device) || !table(a[6], device) || (rot > 0 && (a[5] == Py_None || a[6] == Py_None)))
    Py_RETURN_NONE;
  for (int i : {7, 8, 9})
    if (!ints(THPVariable_Unpack(a[i]), T, device)) Py_RETURN_NONE;
  auto idx = [&](int i) { return THPVariable_Unpack(a[i]).const_data_ptr<int>(); };
  const int rc = append(q.scalar_type() == at::kBFloat16 ? 1 : 2, q.mutable_data_ptr(), k.mutable_data_ptr(), v.const_data_ptr(), q.stride(0),
                        q.stride(1), k.stride(0), k.stride(1), v.stride(0), v.stride(1), T, q.size(1), k.size(1), q.size(2), rot, inter,
                        (const float*)at_or_null(a[5]), (const float*)at_or_null(a[6]), idx(7), idx(8), idx(9), kc.mutable_data_ptr(),
                        vc.mutable_data_ptr(), kc.size(2), stream_of(device));
  return PyBool_FromLong(rc == 0);
  END_HANDLE_TH_ERRORS
}

// packed_attention(q, k, v, cu, max_len, scale, window) -> output, or None: not a call for this function (ALiBi's among them)
PyObject* kca_packed_rows(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 7 || !packed) {
    PyErr_SetString(PyExc_TypeError, "packed_attention(q, k, v, cu, max_len, scale, window) after init_rows");
    return nullptr;
  }
  for (int i : {0, 1, 2, 3})
    if (!is_tensor(a[i])) Py_RETURN_NONE;
  const long max_len = PyLong_AsLong(a[4]), window = PyLong_AsLong(a[6]);
  const double scale = PyFloat_AsDouble(a[5]);
  if (PyErr_Occurred()) return nullptr;
  if (!plain_inference()) Py_RETURN_NONE;
  const Tensor &q = THPVariable_Unpack(a[0]), &k = THPVariable_Unpack(a[1]), &v = THPVariable_Unpack(a[2]), &cu = THPVariable_Unpack(a[3]);
  if (!q.is_cuda() || !half_type(q) || q.dim() != 3) Py_RETURN_NONE;
  const int64_t device = q.get_device(), T = q.size(0), H = q.size(1), D = q.size(2), seqs = cu.numel() - 1;
  if (device != c10::hip::current_device() || !prompt_rows(q, q, device) || !prompt_rows(k, q, device) || !prompt_rows(v, q, device) ||
      k.size(1) != v.size(1) || D % 8 || D > 256 || seqs < 1 || max_len < 1 || !ints(cu, seqs + 1, device))
    Py_RETURN_NONE;
  const bool f16 = q.scalar_type() == at::kHalf;
  Tensor o = at::empty({T, H, D}, q.options()), flags;
  if (!f16) flags = at::empty({4 * ((max_len + 127) / 128) * seqs * H}, cu.options());
  const int rc = packed(f16 ? 2 : 1, q.const_data_ptr(), k.const_data_ptr(), v.const_data_ptr(), o.mutable_data_ptr(), q.stride(0), q.stride(1),
                        k.stride(0), k.stride(1), v.stride(0), v.stride(1), o.stride(0), o.stride(1), seqs, max_len, H, k.size(1), D, 1,
                        (float)scale, nullptr, window, cu.const_data_ptr<int>(), f16 ? nullptr : flags.mutable_data_ptr<int>(),
                        stream_of(device));
  TORCH_CHECK(rc == 0, "kca_attn_fwd_packed returned status ", rc, " (unsupported shape/arguments)");
  return THPVariable_Wrap(std::move(o));
  END_HANDLE_TH_ERRORS
}

// init_rows(kca_rows_mm_two, kca_layernorm_fwd, kca_ln_rows_f16, kca_rope_append, kca_attn_fwd_packed: addresses, counters)
PyObject* kca_init_rows(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 6) {
    PyErr_SetString(PyExc_TypeError, "init_rows(rows_mm_two, layernorm_fwd, ln_rows_f16, rope_append, attn_fwd_packed, counters)");
    return nullptr;
  }
  void* f[5];
  for (int i = 0; i < 5; ++i) f[i] = PyLong_AsVoidPtr(a[i]);
  if (PyErr_Occurred()) return nullptr;
  Py_INCREF(a[5]);
  Py_XSETREF(counters, a[5]);
  rows_mm = reinterpret_cast<RowsFn>(f[0]);
  norm = reinterpret_cast<NormFn>(f[1]);
  norm_f16 = reinterpret_cast<NormF16Fn>(f[2]);
  append = reinterpret_cast<AppendFn>(f[3]);
  packed = reinterpret_cast<PackedFn>(f[4]);
  Py_RETURN_NONE;
}
