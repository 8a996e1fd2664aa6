// Host side of one forward call on torch tensors: the checks of ForwardPlan and gq_linear.forward, the output, the
// workspace and the C struct in native code, then the C entry point whose address the caller hands in.  Host code only; nothing is kept
// from one call for the next.  The steps take 14 to 16 us in Python beside the 7 us of the entry point's two launches, 4 to 6 here, and a decode
// call's kernels 11 to 17: 2560 -> 6144, one row, 4 adapters of rank 64 23.3 -> 12.4 us a call; 12288 -> 4096, 16 rows, 4-bit codes 25.2 -> 18.1.
//
// Both functions return the output tensor, an int (the entry point's status, not OK), or None for anything out of the ordinary -- a wrong
// dtype, shape or device, a tensor subclass or mode, a tensor that is not contiguous, one that requires a gradient, a geometry that
// the library refuses -- and the caller then goes the general way, which converts, differentiates or raises.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/TensorSubclassLikeUtils.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/core/impl/VirtualGuardImpl.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/mi355_w8a8.h"

namespace {

constexpr int64_t kMaxRank = 64, kMaxAdapters = 64;

struct Args {
  PyObject* const* p;
  bool ok = true;
  // an ordinary tensor, or null where the argument is None
  const at::Tensor* tensor(int i) {
    if (p[i] == Py_None) return nullptr;
    if (!THPVariable_CheckExact(p[i])) { ok = false; return nullptr; }
    return &THPVariable_Unpack(p[i]);
  }
  int64_t integer(int i) {
    const int64_t v = PyLong_AsLongLong(p[i]);
    if (v == -1 && PyErr_Occurred()) { PyErr_Clear(); ok = false; }
    return v;
  }
  void* address(int i) { return reinterpret_cast<void*>(static_cast<uintptr_t>(integer(i))); }
};

bool plain(const at::Tensor& t, at::ScalarType type, c10::Device device) {
  return t.layout() == at::kStrided && !t.is_nested() && t.scalar_type() == type && t.device() == device && t.is_contiguous() && t.unsafeGetTensorImpl()->has_storage() &&
         !at::isTensorSubclassLike(t) && !(c10::GradMode::is_enabled() && t.requires_grad());
}

// Rows of K from x; 0 where the call is not an ordinary one.
int64_t rows_of(const at::Tensor* x, int64_t k, int64_t min_dim) {
  if (!x || !x->is_cuda() || x->layout() != at::kStrided || x->is_nested() || x->dim() < min_dim || k <= 0 || x->size(-1) != k || x->numel() == 0) return 0;
  if (c10::impl::TorchDispatchModeTLS::any_modes_set() || !plain(*x, at::kBFloat16, x->device())) return 0;
  if (c10::impl::VirtualGuardImpl(c10::DeviceType::CUDA).getDevice() != x->device()) return 0;
  const int64_t rows = x->numel() / k;
  return rows <= 0x7fffffff ? rows : 0;
}

struct Lora {
  int64_t adapters = 0, rank = 0;
  const void *a = nullptr, *b = nullptr;
  const float* scaling = nullptr;
};
// A [(n,) K, r], B [(n,) r, N], scaling float32 [n]; false where they are not plain or do not fit.
bool lora_of(const at::Tensor* a, const at::Tensor* b, const at::Tensor* s, int64_t k, int64_t n, c10::Device device, Lora& l) {
  if (!a && !b) return true;
  if (!a || !b || !s || a->dim() != b->dim() || (a->dim() != 2 && a->dim() != 3)) return false;
  if (!plain(*a, at::kBFloat16, device) || !plain(*b, at::kBFloat16, device) || !plain(*s, at::kFloat, device)) return false;
  l.adapters = a->dim() == 3 ? a->size(0) : 1;
  l.rank = a->size(-1);
  if (l.adapters < 1 || l.adapters > kMaxAdapters || l.rank < 1 || l.rank > kMaxRank || a->size(-2) != k || b->size(-2) != l.rank || b->size(-1) != n ||
      (b->dim() == 3 && b->size(0) != l.adapters) || s->dim() != 1 || s->size(0) != l.adapters)
    return false;
  l.a = a->const_data_ptr();
  l.b = b->const_data_ptr();
  l.scaling = s->const_data_ptr<float>();
  return true;
}

// Allocations and launches may wait for the GPU: other Python threads go on meanwhile.
struct WithoutGil {
  PyThreadState* const state = PyEval_SaveThread();
  ~WithoutGil() { PyEval_RestoreThread(state); }
};

PyObject* finish(at::Tensor&& out, int status) {
  return status == 0 ? THPVariable_Wrap(std::move(out)) : PyLong_FromLong(status);
}

// dense(x, packed, scales, k, n, a, b, scaling, adapter_indices, gamma, residual, flags, eps, entry, workspace_bytes, forward_path,
// stream)
PyObject* dense(PyObject*, PyObject* const* argv, Py_ssize_t argc) {
  if (argc != 17) { PyErr_SetString(PyExc_TypeError, "dense takes 17 arguments"); return nullptr; }
  HANDLE_TH_ERRORS
  Args arg{argv};
  const at::Tensor *x = arg.tensor(0), *packed = arg.tensor(1), *scales = arg.tensor(2), *a = arg.tensor(5), *b = arg.tensor(6),
                   *s = arg.tensor(7), *idx = arg.tensor(8), *gamma = arg.tensor(9), *residual = arg.tensor(10);
  const int64_t k = arg.integer(3), n = arg.integer(4), flags = arg.integer(11);
  const double eps = PyFloat_Check(argv[12]) ? PyFloat_AS_DOUBLE(argv[12]) : -1.0;
  const auto entry = reinterpret_cast<int (*)(const mi355_w8a8_problem*, void*)>(arg.address(13));
  const auto bytes_of = reinterpret_cast<uint64_t (*)(uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t)>(arg.address(14));
  const auto path_of = reinterpret_cast<int (*)(uint32_t, uint32_t, uint32_t, uint32_t)>(arg.address(15));
  void* const stream = arg.address(16);
  if (!arg.ok || !entry || !bytes_of || !path_of || !packed || !scales || n <= 0 || eps < 0.0) Py_RETURN_NONE;
  const int64_t m = rows_of(x, k, 2);
  if (m == 0) Py_RETURN_NONE;
  const c10::Device device = x->device();
  if (!plain(*packed, at::kByte, device) || !plain(*scales, at::kFloat, device)) Py_RETURN_NONE;
  Lora lora;
  if (!lora_of(a, b, s, k, n, device, lora)) Py_RETURN_NONE;
  const bool swiglu = (flags & MI355_W8A8_FLAG_SWIGLU) != 0;
  if (swiglu && n % 2) Py_RETURN_NONE;
  at::DimVector shape(x->sizes().begin(), x->sizes().end());
  shape.back() = swiglu ? n / 2 : n;
  if (gamma && (!plain(*gamma, at::kFloat, device) || gamma->dim() != 1 || gamma->size(0) != k)) Py_RETURN_NONE;
  if (residual && (!plain(*residual, at::kBFloat16, device) || residual->sizes() != at::IntArrayRef(shape))) Py_RETURN_NONE;
  if (idx && (!lora.adapters || !plain(*idx, at::kInt, device) || idx->numel() == 0 || m % idx->numel())) Py_RETURN_NONE;
  const uint64_t bytes = bytes_of((uint32_t)m, (uint32_t)k, (uint32_t)n, (uint32_t)lora.adapters, (uint32_t)lora.rank, (uint32_t)flags);
  if (bytes == 0) Py_RETURN_NONE;
  at::Tensor out;
  int status;
  {
    const WithoutGil released;
    // One index per example, whose rows follow each other: the routing launch of the tiled paths reads it as it is (the decode
    // kernels take an index per row, and every path an aligned array).
    at::Tensor rows_idx;
    uint32_t per = 1;
    if (idx) {
      rows_idx = *idx;
      const int64_t rows = m / idx->numel();
      if (rows > 1) {
        const int path = path_of((uint32_t)m, (uint32_t)k, (uint32_t)n, (uint32_t)flags);
        if (path == MI355_W8A8_PATH_SKINNY || path == MI355_W8A8_PATH_SKINNY_CHUNKS || (reinterpret_cast<uintptr_t>(idx->const_data_ptr()) & 15u))
          rows_idx = idx->reshape({-1, 1}).expand({idx->numel(), rows}).contiguous();
        else
          per = (uint32_t)rows;
      }
    }
    out = at::empty(shape, x->options().requires_grad(false));
    const at::Tensor ws = at::empty({(int64_t)bytes}, packed->options().requires_grad(false));
    mi355_w8a8_problem_z whole{};
    whole.rows_per_index = per;
    mi355_w8a8_problem& p = whole.call;
    p.struct_size = sizeof(whole);
    p.flags = (uint32_t)flags;
    p.m = (uint32_t)m; p.k = (uint32_t)k; p.n = (uint32_t)n;
    p.n_adapters = (uint32_t)lora.adapters; p.rank = (uint32_t)lora.rank;
    p.rms_eps = (float)eps;
    p.x = x->const_data_ptr();
    p.w_packed = packed->const_data_ptr(); p.w_scales = scales->const_data_ptr<float>();
    p.lora_a = lora.a; p.lora_b = lora.b; p.lora_scaling = lora.scaling;
    p.adapter_indices = idx ? rows_idx.const_data_ptr<int32_t>() : nullptr;
    p.rms_gamma = gamma ? gamma->const_data_ptr<float>() : nullptr;
    p.residual = residual ? residual->const_data_ptr() : nullptr;
    p.out = out.mutable_data_ptr();
    p.workspace = ws.mutable_data_ptr();
    p.workspace_bytes = bytes;
    // (what the kernels touch was allocated for the stream they are enqueued on, or is held by the caller)
    status = entry(&p, stream);
  }
  return finish(std::move(out), status);
  END_HANDLE_TH_ERRORS
}

// group_scaled(x, packed, scales, k, k_pad, n, group, weight_bits, activation_bits, a, b, scaling, entry, workspace_bytes, stream)
PyObject* group_scaled(PyObject*, PyObject* const* argv, Py_ssize_t argc) {
  if (argc != 15) { PyErr_SetString(PyExc_TypeError, "group_scaled takes 15 arguments"); return nullptr; }
  HANDLE_TH_ERRORS
  Args arg{argv};
  const at::Tensor *x = arg.tensor(0), *packed = arg.tensor(1), *scales = arg.tensor(2), *a = arg.tensor(9), *b = arg.tensor(10),
                   *s = arg.tensor(11);
  const int64_t k = arg.integer(3), k_pad = arg.integer(4), n = arg.integer(5), group = arg.integer(6), wbits = arg.integer(7),
                abits = arg.integer(8);
  const auto entry = reinterpret_cast<int (*)(const mi355_w8a8_gq_problem*, void*)>(arg.address(12));
  const auto bytes_of = reinterpret_cast<uint64_t (*)(uint32_t, uint32_t, uint32_t, uint32_t, uint32_t)>(arg.address(13));
  void* const stream = arg.address(14);
  if (!arg.ok || !entry || !bytes_of || !packed || !scales || n <= 0 || k_pad <= 0 || group <= 0) Py_RETURN_NONE;
  const int64_t m = rows_of(x, k, 1);
  if (m == 0) Py_RETURN_NONE;
  const c10::Device device = x->device();
  if (!plain(*packed, at::kByte, device) || !plain(*scales, at::kFloat, device)) Py_RETURN_NONE;
  Lora lora;
  if (!lora_of(a, b, s, k, n, device, lora)) Py_RETURN_NONE;
  const uint64_t bytes = bytes_of((uint32_t)m, (uint32_t)k_pad, (uint32_t)group, (uint32_t)lora.adapters, (uint32_t)lora.rank);
  if (bytes == 0) Py_RETURN_NONE;
  at::DimVector shape(x->sizes().begin(), x->sizes().end());
  shape.back() = n;
  at::Tensor out;
  int status;
  {
    const WithoutGil released;
    out = at::empty(shape, x->options().requires_grad(false));
    const at::Tensor ws = at::empty({(int64_t)bytes}, packed->options().requires_grad(false));
    mi355_w8a8_gq_problem p{};
    p.struct_size = sizeof(p);
    p.m = (uint32_t)m; p.k = (uint32_t)k; p.k_pad = (uint32_t)k_pad; p.n = (uint32_t)n;
    p.group_size = (uint32_t)group; p.weight_bits = (uint32_t)wbits; p.activation_bits = (uint32_t)abits;
    p.n_adapters = (uint32_t)lora.adapters; p.rank = (uint32_t)lora.rank;
    p.x = x->const_data_ptr();
    p.w_packed = packed->const_data_ptr(); p.w_scales = scales->const_data_ptr<float>();
    p.lora_a = lora.a; p.lora_b = lora.b; p.lora_scaling = lora.scaling;
    p.out = out.mutable_data_ptr();
    p.workspace = ws.mutable_data_ptr();
    p.workspace_bytes = bytes;
    status = entry(&p, stream);
  }
  return finish(std::move(out), status);
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"dense", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(dense)), METH_FASTCALL, "One forward call of the per-channel linear."},
    {"group_scaled", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(group_scaled)), METH_FASTCALL,
     "One forward call of the group-scaled linear."},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "mi355_w8a8_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_mi355_w8a8_host() {
  PyObject* const m = PyModule_Create(&module);
  if (m && PyModule_AddStringConstant(m, "torch_version", MI355_TORCH_VERSION) != 0) {  // (its C++ ABI is this one's: _native.host)
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
