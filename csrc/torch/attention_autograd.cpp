// flash_attention as an autograd function without Python frames: argument checks, allocations, kernel launches and the node of
// the backward pass in C++ (ops/attention.py holds the same function in Python, which every call that is not plain eager
// work on plain tensors still takes).
//
// Why: a short training call is bound by the host. 1 x 96 tokens x 12 heads of 64, forward and backward, is 20 us of kernels
// that took 132 us to issue: ctypes converts 33 and 45 arguments (25 us), and the backward pass waits for the interpreter
// lock in the engine's thread.
#include "prompt_rows.h"

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;
typedef long long ll;

// kca_attn_fwd, kca_attn_bwd of the kernel library that ops/_lib.py has loaded
typedef int (*FwdFn)(const void*, const void*, const void*, void*, float*, ll, ll, ll, ll, ll, ll, ll, ll, ll, ll, ll, ll, int, int,
                     int, int, int, int, int, float, const float*, const int*, int, const unsigned*, int, int, int*, hipStream_t);
typedef int (*BwdFn)(const void*, const void*, const void*, const void*, const void*, void*, void*, void*, const float*, float*, ll,
                     ll, ll, ll, ll, ll, ll, ll, ll, ll, ll, ll, ll, ll, ll, ll, ll, ll, ll, ll, ll, ll, ll, ll, int, int, int, int,
                     int, int, int, float, const float*, const int*, int, const unsigned*, hipStream_t);
FwdFn attn_fwd = nullptr;
BwdFn attn_bwd = nullptr;

#define STRIDES(t) (t).stride(0), (t).stride(1), (t).stride(2)

// the kernels' mask arguments: int32 lengths [B] or a bitmap [B, W]
const int* lengths(const std::optional<Tensor>& m) { return m && m->dim() == 1 ? m->const_data_ptr<int>() : nullptr; }
const unsigned* bitmap(const std::optional<Tensor>& m) {
  return m && m->dim() != 1 ? reinterpret_cast<const unsigned*>(m->const_data_ptr<int>()) : nullptr;
}
const float* slopes(const std::optional<Tensor>& a) { return a ? a->const_data_ptr<float>() : nullptr; }
hipStream_t stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.get_device()).stream(); }

struct FlashAttn : torch::autograd::Function<FlashAttn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, bool causal, double scale,
                        const std::optional<Tensor>& mask, const std::optional<Tensor>& alibi, int64_t window) {
    const int64_t B = q.size(0), Sq = q.size(1), H = q.size(2), D = q.size(3), Sk = k.size(1), Hkv = k.size(2);
    Tensor o = at::empty({B, Sq, H, D}, q.options());
    // log-sum-exp of the rows, and behind it the overflow flags of the kernels that have some (4 a 128-row block)
    const int64_t rows = B * H * Sq, flags = 4 * ((Sq + 127) / 128) * B * H;
    Tensor lse = at::empty({rows + flags}, q.options().dtype(at::kFloat));
    float* l = lse.mutable_data_ptr<float>();
    const int rc = attn_fwd(q.const_data_ptr(), k.const_data_ptr(), v.const_data_ptr(), o.mutable_data_ptr(), l, STRIDES(q),
                            STRIDES(k), STRIDES(v), STRIDES(o), B, Sq, Sk, H, Hkv, D, causal, (float)scale, slopes(alibi),
                            lengths(mask), window, bitmap(mask), -1, -1, reinterpret_cast<int*>(l + rows), stream_of(q));
    TORCH_CHECK(rc == 0, "kca_attn_fwd returned status ", rc, " (unsupported shape/arguments)");
    ctx->save_for_backward({q, k, v, o, lse, mask.value_or(Tensor()), alibi.value_or(Tensor())});
    ctx->saved_data["causal"] = causal;
    ctx->saved_data["scale"] = scale;
    ctx->saved_data["window"] = window;
    return o;
  }

  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    const variable_list saved = ctx->get_saved_variables();
    const Tensor &q = saved[0], &k = saved[1], &v = saved[2], &o = saved[3], &lse = saved[4];
    auto given = [](const Tensor& t) { return t.defined() ? std::optional<Tensor>(t) : std::nullopt; };
    const auto mask = given(saved[5]), alibi = given(saved[6]);
    const c10::OptionalDeviceGuard guard(q.device());
    const Tensor g = grads[0].contiguous();
    const int64_t B = q.size(0), Sq = q.size(1), H = q.size(2), D = q.size(3), Sk = k.size(1), Hkv = k.size(2);
    Tensor dq = at::empty(q.sizes(), q.options()), dk = at::empty(k.sizes(), k.options()), dv = at::empty(v.sizes(), v.options());
    Tensor delta = at::empty({B * H * Sq}, lse.options());
    const int rc = attn_bwd(q.const_data_ptr(), k.const_data_ptr(), v.const_data_ptr(), o.const_data_ptr(), g.const_data_ptr(),
                            dq.mutable_data_ptr(), dk.mutable_data_ptr(), dv.mutable_data_ptr(), lse.const_data_ptr<float>(),
                            delta.mutable_data_ptr<float>(), STRIDES(q), STRIDES(k), STRIDES(v), STRIDES(o), STRIDES(g), STRIDES(dq),
                            STRIDES(dk), STRIDES(dv), B, Sq, Sk, H, Hkv, D, ctx->saved_data["causal"].toBool(),
                            (float)ctx->saved_data["scale"].toDouble(), slopes(alibi), lengths(mask),
                            ctx->saved_data["window"].toInt(), bitmap(mask), stream_of(q));
    TORCH_CHECK(rc == 0, "kca_attn_bwd returned status ", rc, " (unsupported shape/arguments)");
    return {dq, dk, dv, Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

// No transform, mode, trace or tangent that a Python autograd function would see and this one would not.
bool plain_state() {
  return !c10::impl::TorchDispatchModeTLS::any_modes_set() && !at::impl::torch_function_mode_enabled() &&
         !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) &&
         !torch::jit::tracer::isTracing();
}

bool kernel_input(const Tensor& t, int64_t device) {
  return t.dim() == 4 && t.stride(3) == 1 && t.scalar_type() == at::kBFloat16 && t.layout() == at::kStrided &&
         t.get_device() == device && !t._fw_grad(0).defined();
}

// attention(q, k, v, causal, scale, mask | None, alibi | None, window) -> output, or None: not a call for this function
PyObject* attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 8 || !attn_fwd) {
    PyErr_SetString(PyExc_TypeError, "attention(q, k, v, causal, scale, mask, alibi, window) after init");
    return nullptr;
  }
  for (int i : {0, 1, 2, 5, 6})
    if (!THPVariable_CheckExact(a[i]) && !(i > 4 && a[i] == Py_None)) Py_RETURN_NONE;
  if (!plain_state()) Py_RETURN_NONE;
  const Tensor &q = THPVariable_Unpack(a[0]), &k = THPVariable_Unpack(a[1]), &v = THPVariable_Unpack(a[2]);
  if (!q.is_cuda()) Py_RETURN_NONE;
  const int64_t device = q.get_device();
  if (device != c10::hip::current_device() || !kernel_input(q, device) || !kernel_input(k, device) || !kernel_input(v, device) ||
      q.size(3) % 8 || q.size(3) > 256)
    Py_RETURN_NONE;
  std::optional<Tensor> mask, alibi;
  if (a[5] != Py_None) mask = THPVariable_Unpack(a[5]);
  if (a[6] != Py_None) alibi = THPVariable_Unpack(a[6]);
  if ((mask && (mask->scalar_type() != at::kInt || mask->get_device() != device)) ||
      (alibi && (alibi->scalar_type() != at::kFloat || alibi->get_device() != device || alibi->requires_grad())))
    Py_RETURN_NONE;
  const int causal = PyObject_IsTrue(a[3]);
  const double scale = PyFloat_AsDouble(a[4]);
  const long window = PyLong_AsLong(a[7]);
  if (causal < 0 || PyErr_Occurred()) return nullptr;
  return THPVariable_Wrap(FlashAttn::apply(q, k, v, causal != 0, scale, mask, alibi, (int64_t)window));
  END_HANDLE_TH_ERRORS
}

// init(address of kca_attn_fwd, address of kca_attn_bwd)
PyObject* init(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 2) {
    PyErr_SetString(PyExc_TypeError, "init(forward, backward)");
    return nullptr;
  }
  void *f = PyLong_AsVoidPtr(a[0]), *b = PyLong_AsVoidPtr(a[1]);
  if (PyErr_Occurred()) return nullptr;
  attn_bwd = reinterpret_cast<BwdFn>(b);
  attn_fwd = reinterpret_cast<FwdFn>(f);
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {{"attention", (PyCFunction)(void (*)())attention, METH_FASTCALL, nullptr},
                         {"init", (PyCFunction)(void (*)())init, METH_FASTCALL, nullptr},
                         {"few_rows", (PyCFunction)(void (*)())kca_few_rows, METH_FASTCALL, nullptr},
                         {"norm_rows", (PyCFunction)(void (*)())kca_norm_rows, METH_FASTCALL, nullptr},
                         {"rope_append", (PyCFunction)(void (*)())kca_rope_rows, METH_FASTCALL, nullptr},
                         {"packed_attention", (PyCFunction)(void (*)())kca_packed_rows, METH_FASTCALL, nullptr},
                         {"init_rows", (PyCFunction)(void (*)())kca_init_rows, METH_FASTCALL, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module{PyModuleDef_HEAD_INIT, "kca_torch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// `torch`: the version that it was compiled against, whose class layouts are in it (ops/_lib.py looks before it uses the module)
PyMODINIT_FUNC PyInit_kca_torch() {
  PyObject* m = PyModule_Create(&module);
  if (m && PyModule_AddStringConstant(m, "torch", KCA_TORCH) < 0) Py_CLEAR(m);
  return m;
}
