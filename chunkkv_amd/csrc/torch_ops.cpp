// The torch-facing calls that a decoder layer makes many times per request, as one CPython call
// each: argument checks, output allocation and the C-ABI launch (include/chunkkv_amd.h) without the
// interpreter in between. chunkkv_amd/ops.py keeps their names, signatures and documentation and
// raises the same exceptions for the same misuse; everything else there calls the C ABI through
// ctypes.
//
// Bound: host time. A layer's launches take 3-15 us on the GPU at short requests, and a wrapper in
// Python (a dozen tensor attributes, an allocation, a 20-argument ctypes call) took 8-11 us of the
// host for each: attention_active 9.4 us, rope_qkv (k/v into a cache) 10.9, add_rmsnorm 8.0,
// silu_mul 12.2. The launch itself is 2-3 us of that.
#include <Python.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>
#include <torch/types.h>
#include <pybind11/pybind11.h>

#include <algorithm>
#include <cmath>
#include <string>
#include <utility>
#include <vector>

#include "chunkkv_amd.h"

namespace {

using at::Tensor;

// A Python exception on its way out: ValueError, TypeError or RuntimeError with a message.
struct PyFailure {
  PyObject* type;
  std::string what;
};
[[noreturn]] void value_error(std::string s) { throw PyFailure{PyExc_ValueError, std::move(s)}; }
[[noreturn]] void type_error(std::string s) { throw PyFailure{PyExc_TypeError, std::move(s)}; }

#define CKV_PY_BEGIN HANDLE_TH_ERRORS try {
#define CKV_PY_END                          \
  }                                         \
  catch (const PyFailure& f) {              \
    PyErr_SetString(f.type, f.what.c_str()); \
    return nullptr;                         \
  }                                         \
  END_HANDLE_TH_ERRORS

void need_args(Py_ssize_t got, Py_ssize_t want) {
  if (got != want) type_error("expected " + std::to_string(want) + " arguments, got " + std::to_string(got));
}
const Tensor& tensor(PyObject* o) {
  if (!THPVariable_Check(o)) type_error(std::string("expected a tensor, got ") + Py_TYPE(o)->tp_name);
  return THPVariable_Unpack(o);
}
Tensor optional_tensor(PyObject* o) { return o == Py_None ? Tensor() : tensor(o); }
int64_t integer(PyObject* o) {
  const int64_t v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) throw python_error();
  return v;
}
double real(PyObject* o) {
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) throw python_error();
  return v;
}
int32_t int32(int64_t v) { return (int32_t)v; }  // as a ctypes c_int32 argument takes it

void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
void* stream_of(const Tensor& t) {
  return (void*)c10::hip::getCurrentHIPStream(t.device().index()).stream();
}
int dtype_code(const Tensor& t) {
  if (t.scalar_type() == at::kBFloat16) return CKV_DTYPE_BF16;
  if (t.scalar_type() == at::kFloat) return CKV_DTYPE_F32;
  type_error(std::string("unsupported K/V dtype ") + c10::toString(t.scalar_type()) +
             "; the HIP kernels take float32 or bfloat16");
}

// Every tensor on one HIP device.
template <typename... T>
void same_device(const Tensor& first, const T&... rest) {
  for (const Tensor* t : {&first, &rest...}) {
    if (!t->is_cuda()) value_error("chunkkv_amd ops run on a HIP device; got a tensor on " + t->device().str());
    if (t->device() != first.device())
      value_error("tensors on different devices: " + t->device().str() + " vs " + first.device().str());
  }
}
void need_dims(const Tensor& t, int64_t d, const char* what) {
  if (t.dim() != d) value_error(std::string(what) + " must have " + std::to_string(d) + " dimensions");
}
std::string shape_of(const Tensor& t) {
  std::string s = "(";
  for (int64_t i = 0; i < t.dim(); ++i) s += (i ? ", " : "") + std::to_string(t.size(i));
  return s + ")";
}
// Last dim contiguous, base and every other stride on a 16-byte boundary; else a contiguous copy.
Tensor rows_view(const Tensor& t) {
  bool ok = t.stride(-1) == 1 && (uintptr_t)t.data_ptr() % 16 == 0;
  for (int64_t i = 0; i + 1 < t.dim(); ++i) ok = ok && t.stride(i) * t.element_size() % 16 == 0;
  return ok ? t : t.contiguous();
}

// The status of a C-ABI call as the exception chunkkv_amd/_native.py:check raises.
void check(int32_t status, const char* what) {
  if (status == CKV_OK) return;
  const std::string msg =
      std::string(what) + ": " + ckv_status_string(status) + " (status " + std::to_string(status) + ")";
  if (status == CKV_ERR_INVALID_ARGUMENT || status == CKV_ERR_OUT_OF_RANGE || status == CKV_ERR_TOO_LARGE) value_error(msg);
  throw PyFailure{PyExc_RuntimeError, msg};
}
// The launch itself runs without the interpreter lock, as a ctypes call does. f looks up addresses
// and the stream too, which throw (a tensor without storage, a HIP error): the lock is taken back
// on that way out as well, before any handler touches the interpreter.
struct Unlocked {
  PyThreadState* const state = PyEval_SaveThread();
  Unlocked() = default;
  Unlocked(const Unlocked&) = delete;
  Unlocked& operator=(const Unlocked&) = delete;
  ~Unlocked() { PyEval_RestoreThread(state); }
};
template <typename F>
int32_t unlocked(F f) {
  const Unlocked section;
  return f();
}

// attention_active(q, K, V, positions, scale, err, out, split)
PyObject* attention_active(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  CKV_PY_BEGIN
  need_args(n_args, 8);
  Tensor q = tensor(a[0]);
  const Tensor &K = tensor(a[1]), &V = tensor(a[2]);
  Tensor pos = tensor(a[3]);
  const Tensor err = optional_tensor(a[5]);
  Tensor out = optional_tensor(a[6]);
  same_device(q, K, V, pos);
  need_dims(q, 4, "q");
  need_dims(K, 4, "K");
  const int64_t Hq = q.size(1), n = q.size(2), D = q.size(3), Hkv = K.size(1), N = K.size(2);
  if (q.scalar_type() != at::kBFloat16 || K.scalar_type() != at::kBFloat16 || V.scalar_type() != at::kBFloat16)
    type_error("attention_active runs on bf16 q/K/V");
  if (!K.is_contiguous() || !V.is_contiguous() || V.sizes() != K.sizes() || K.size(3) != D)
    value_error("K/V must be contiguous (1, Hkv, N, D) and match q's head_dim");
  if (q.stride(3) != 1) q = q.contiguous();
  if (pos.scalar_type() != at::kLong || pos.numel() != n) value_error("positions must be int64 (n,)");
  pos = pos.contiguous();
  if (!out.defined()) {
    out = at::empty({1, n, Hq, D}, q.options());
  } else if (out.sizes() != at::IntArrayRef({1, n, Hq, D}) || !out.is_contiguous() || out.scalar_type() != q.scalar_type()) {
    value_error("out must be contiguous (1, n, Hq, D) bf16");
  }
  const double scale = a[4] == Py_None ? 1.0 / std::sqrt((double)D) : real(a[4]);
  const int split = PyObject_IsTrue(a[7]);
  if (split < 0) throw python_error();
  const int64_t ws_bytes =
      split ? ckv_attention_workspace_bytes(int32(n), int32(N), int32(Hq), int32(D), nullptr, nullptr) : 0;
  Tensor ws;
  if (ws_bytes > 0) ws = at::empty({ws_bytes / 4}, q.options().dtype(at::kFloat));
  check(unlocked([&] {
          return ckv_attention_active(ptr(out), ptr(q), q.stride(1), q.stride(2), ptr(K), ptr(V), N * D,
                                      (const int64_t*)ptr(pos), int32(n), int32(N), int32(Hq), int32(Hkv), int32(D),
                                      CKV_DTYPE_BF16, scale, ptr(ws), ws_bytes, (int32_t*)ptr(err), stream_of(q));
        }),
        "ckv_attention_active");
  return THPVariable_Wrap(out);
  CKV_PY_END
}

// Pointer, head stride and token stride of a (1, n, n_heads * D) token-major tensor or a
// (1, H, n, D) tensor with contiguous rows.
struct Heads {
  void* p = nullptr;
  int64_t hs = 0, ts = 0;
};
Heads heads_view(const Tensor& t, int64_t n_heads, int64_t D) {
  if (t.dim() == 3) {
    if (t.stride(2) != 1 || t.size(2) != n_heads * D)
      value_error("projection output must have contiguous rows of n_heads * head_dim");
    return {ptr(t), D, t.stride(1)};
  }
  if (t.dim() == 4 && t.size(1) == n_heads && t.size(3) == D && t.stride(3) == 1) return {ptr(t), t.stride(1), t.stride(2)};
  value_error("unsupported layout " + shape_of(t));
}

// rope_qkv(q_in, k_in, v_in, positions, n_q_heads, n_kv_heads, head_dim, theta, q_out, k_out, v_out, rows, table, err)
PyObject* rope_qkv(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  CKV_PY_BEGIN
  need_args(n_args, 14);
  const Tensor &k_in = tensor(a[1]), v_in = optional_tensor(a[2]);
  Tensor pos = tensor(a[3]);
  const int64_t Hq = integer(a[4]), Hkv = integer(a[5]), D = integer(a[6]);
  const double theta = real(a[7]);
  const Tensor q_in = Hq == 0 ? k_in : tensor(a[0]);  // k/v only: q is not read
  Tensor q_out = optional_tensor(a[8]), k_out = optional_tensor(a[9]);
  const Tensor v_out = optional_tensor(a[10]), table = optional_tensor(a[12]), err = optional_tensor(a[13]);
  Tensor rows = optional_tensor(a[11]);
  if (table.defined()) {
    same_device(k_in, table);
    if (table.scalar_type() != at::kFloat || table.dim() != 3 || table.size(1) != D / 2 || table.size(2) != 2)
      value_error("table must be a rope_table() output (n, D/2, 2) float32");
  }
  same_device(k_in, pos);
  const int64_t n = pos.numel();
  if (pos.scalar_type() != at::kLong) value_error("positions must be int64");
  const bool rows_are_positions = rows.defined() && a[11] == a[3];
  pos = pos.contiguous();
  if (!q_out.defined() && Hq) q_out = at::empty({1, n, Hq, D}, q_in.options().device(k_in.device()));
  if (!k_out.defined()) {
    if (rows.defined()) value_error("rows needs k_out (the cache)");
    k_out = at::empty({1, Hkv, n, D}, q_in.options().device(k_in.device()));
  }
  const int64_t n_out = k_out.dim() == 4 ? k_out.size(2) : k_out.size(1);
  if (rows.defined()) {
    same_device(q_in, rows);
    if (rows.scalar_type() != at::kLong || rows.numel() != n) value_error("rows must be int64 (n,)");
    rows = rows_are_positions ? pos : rows.contiguous();
  }
  if (v_in.defined() != v_out.defined()) value_error("v_in and v_out go together");
  const auto dt = q_in.scalar_type();
  if (k_in.scalar_type() != dt || k_out.scalar_type() != dt || (Hq && q_out.scalar_type() != dt) ||
      (v_in.defined() && (v_in.scalar_type() != dt || v_out.scalar_type() != dt)))
    type_error("q/k/v and outputs must share a dtype");
  Heads qo, qi, vi, vo;
  if (Hq) {
    if (q_out.sizes() != at::IntArrayRef({1, n, Hq, D}) || !q_out.is_contiguous())
      value_error("q_out must be contiguous (1, n, Hq, D), token-major");
    qo = {ptr(q_out), D, Hq * D};
    qi = heads_view(q_in, Hq, D);
  }
  const Heads ki = heads_view(k_in, Hkv, D), ko = heads_view(k_out, Hkv, D);
  if (v_in.defined()) vi = heads_view(v_in, Hkv, D);
  if (v_out.defined()) vo = heads_view(v_out, Hkv, D);
  const int code = dtype_code(q_in);
  check(unlocked([&] {
          return ckv_rope_qkv(qo.p, qo.hs, qo.ts, ko.p, ko.hs, ko.ts, vo.p, vo.hs, vo.ts, (const int64_t*)ptr(rows),
                              int32(n_out), qi.p, qi.hs, qi.ts, ki.p, ki.hs, ki.ts, vi.p, vi.hs, vi.ts,
                              (const int64_t*)ptr(pos), ptr(table), table.defined() ? table.size(0) : 0, int32(n),
                              int32(Hq), int32(Hkv), int32(D), code, theta, (int32_t*)ptr(err), stream_of(k_in));
        }),
        "ckv_rope_qkv");
  PyObject* q_obj;
  if (q_out.defined()) {
    q_obj = THPVariable_Wrap(q_out);
  } else {
    Py_INCREF(Py_None);
    q_obj = Py_None;
  }
  return Py_BuildValue("(NN)", q_obj, THPVariable_Wrap(k_out));
  CKV_PY_END
}

// add_rmsnorm(h, delta, weight, eps, h_out, out)
PyObject* add_rmsnorm(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  CKV_PY_BEGIN
  need_args(n_args, 6);
  const Tensor &h = tensor(a[0]), delta = optional_tensor(a[1]), &weight = tensor(a[2]);
  const double eps = real(a[3]);
  Tensor h_out = optional_tensor(a[4]), out = optional_tensor(a[5]);
  if (delta.defined()) same_device(h, weight, delta);
  else same_device(h, weight);
  if (h.dim() == 0) throw PyFailure{PyExc_IndexError, "tuple index out of range"};
  const int64_t hidden = h.size(-1);
  if (!h.is_contiguous() || (delta.defined() && (!delta.is_contiguous() || delta.sizes() != h.sizes())))
    value_error("h and delta must be contiguous and of one shape");
  if (weight.dim() != 1 || weight.size(0) != hidden || weight.scalar_type() != h.scalar_type() ||
      (delta.defined() && delta.scalar_type() != h.scalar_type()))
    value_error("weight must be (hidden,) and every operand of h's dtype");
  auto fits = [&](const Tensor& t) { return t.sizes() == h.sizes() && t.is_contiguous() && t.scalar_type() == h.scalar_type(); };
  if (!out.defined()) out = at::empty(h.sizes(), h.options());
  else if (!fits(out)) value_error("out must be contiguous, of h's shape and dtype");
  if (delta.defined() && !h_out.defined()) h_out = at::empty(h.sizes(), h.options());
  else if (h_out.defined() && !fits(h_out)) value_error("h_out must be contiguous, of h's shape and dtype");
  const Tensor w = weight.contiguous();
  const int code = dtype_code(h);
  check(unlocked([&] {
          return ckv_add_rmsnorm(ptr(h_out), ptr(h), ptr(delta), ptr(out), ptr(w), hidden ? h.numel() / hidden : 0,
                                 int32(hidden), (float)eps, code, stream_of(h));
        }),
        "ckv_add_rmsnorm");
  return Py_BuildValue("(NN)", THPVariable_Wrap(delta.defined() ? h_out : h), THPVariable_Wrap(out));
  CKV_PY_END
}

// Row stride (elements) of a (..., width) tensor whose rows are contiguous and evenly spaced.
int64_t row_major(const Tensor& t, int64_t width, const char* what) {
  const std::string w(what);
  if (t.size(-1) != width || t.stride(-1) != 1 || (uintptr_t)t.data_ptr() % 16 != 0)
    value_error(w + " must have contiguous, 16-byte aligned rows of " + std::to_string(width) + " elements");
  if (t.dim() == 2) return t.size(0) > 1 ? t.stride(0) : width;
  int64_t step = -1, seen = 1;  // outer dimensions, innermost first: each must continue the ones inside it
  for (int64_t i = t.dim() - 2; i >= 0; --i) {
    if (t.size(i) == 0) return width;
    if (t.size(i) == 1) continue;
    if (step < 0) step = t.stride(i);
    else if (t.stride(i) != step * seen) value_error(w + " rows must be evenly spaced");
    seen *= t.size(i);
  }
  return step < 0 ? width : step;
}

// silu_mul(gate, up, out)
PyObject* silu_mul(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  CKV_PY_BEGIN
  need_args(n_args, 3);
  const Tensor &gate = tensor(a[0]), &up = tensor(a[1]);
  Tensor out = optional_tensor(a[2]);
  same_device(gate, up);
  if (gate.dim() == 0) throw PyFailure{PyExc_IndexError, "tuple index out of range"};
  const int64_t width = gate.size(-1);
  if (up.sizes() != gate.sizes() || up.scalar_type() != gate.scalar_type())
    value_error("gate and up must have one shape and dtype");
  const int64_t gs = row_major(gate, width, "gate"), us = row_major(up, width, "up");
  if (!out.defined()) {
    out = at::empty(gate.sizes(), gate.options());
  } else if (out.sizes() != gate.sizes() || !out.is_contiguous() || out.scalar_type() != gate.scalar_type()) {
    value_error("out must be contiguous, of gate's shape and dtype");
  }
  const int code = dtype_code(gate);
  check(unlocked([&] {
          return ckv_silu_mul(ptr(out), width, ptr(gate), gs, ptr(up), us, width ? gate.numel() / width : 0,
                              int32(width), code, stream_of(gate));
        }),
        "ckv_silu_mul");
  return THPVariable_Wrap(out);
  CKV_PY_END
}

// Whether a call with these operands would reach torch's device code with nothing in between: no
// tracing, transform (vmap), mode, autocast or tensor subclass takes part, which the kernels here
// know nothing of.
bool unintercepted(c10::DispatchKeySet operands) {
  static const c10::DispatchKeySet plain({c10::DispatchKey::CUDA, c10::DispatchKey::AutogradCUDA,
                                          c10::DispatchKey::ADInplaceOrView, c10::DispatchKey::BackendSelect});
  const auto tls = c10::impl::tls_local_dispatch_key_set();
  const c10::DispatchKeySet keys = (operands | tls.included_) - tls.excluded_;
  return (keys.raw_repr() & ~plain.raw_repr()) == 0;
}

// linear(x, weight, bias): ckv_linear where it is the better choice and takes the operands, else torch's
PyObject* linear(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  CKV_PY_BEGIN
  need_args(n_args, 3);
  const Tensor &x = tensor(a[0]), &w = tensor(a[1]), bias = optional_tensor(a[2]);
  auto plain = [&](const Tensor& t) {
    return t.is_cuda() && t.device() == x.device() && t.scalar_type() == at::kBFloat16 && t.is_contiguous() &&
           unintercepted(t.key_set()) && !t._fw_grad(/*level=*/0).defined() && (uintptr_t)t.data_ptr() % 16 == 0 &&
           !(at::GradMode::is_enabled() && t.requires_grad());
  };
  int64_t ws_bytes = -1;
  if (x.dim() >= 2 && w.dim() == 2 && x.size(-1) == w.size(1) && w.numel() > 0 && x.numel() > 0 && plain(x) && plain(w) &&
      (!bias.defined() || (bias.dim() == 1 && bias.size(0) == w.size(0) && plain(bias)))) {
    const int64_t rows = x.numel() / x.size(-1);
    if (rows <= INT32_MAX && w.size(0) <= INT32_MAX && w.size(1) <= INT32_MAX)
      ws_bytes = ckv_linear_workspace_bytes(int32(rows), int32(w.size(0)), int32(w.size(1)));
  }
  if (ws_bytes < 0) {
    Tensor out;
    {
      pybind11::gil_scoped_release off;
      out = at::linear(x, w, bias.defined() ? std::optional<Tensor>(bias) : std::nullopt);
    }
    return THPVariable_Wrap(out);
  }
  at::DimVector shape(x.sizes().begin(), x.sizes().end());
  shape.back() = w.size(0);
  Tensor out = at::empty(shape, x.options()), ws;
  if (ws_bytes > 0) ws = at::empty({ws_bytes / 4}, x.options().dtype(at::kFloat));
  check(unlocked([&] {
          return ckv_linear(ptr(out), ptr(x), x.size(-1), ptr(w), ptr(bias), int32(x.numel() / x.size(-1)),
                            int32(w.size(0)), int32(w.size(1)), CKV_DTYPE_BF16, ptr(ws), ws_bytes, stream_of(x));
        }),
        "ckv_linear");
  return THPVariable_Wrap(out);
  CKV_PY_END
}

// layer1_repair_gather(k_slab, v_slab, src_tab, layer, begin, end, segments, n_segs, max_seg_tokens, k, v, flags,
//                      local, spans, threshold, theta, workspace, err, out, diff_norm) with out None or the six
// tensors of a Selection and diff_norm None or two: (diff, norm, the six tensors)
PyObject* layer1_repair_gather(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  CKV_PY_BEGIN
  need_args(n_args, 20);
  const Tensor &ks = tensor(a[0]), &vs = tensor(a[1]), &tab = tensor(a[2]);
  const int64_t layer = integer(a[3]), begin = integer(a[4]), end = integer(a[5]);
  const Tensor& segs = tensor(a[6]);
  const int64_t n_segs = integer(a[7]), max_seg = integer(a[8]);
  Tensor k = tensor(a[9]), v = tensor(a[10]);
  const Tensor &flags = tensor(a[11]), &local = tensor(a[12]), &spans = tensor(a[13]);
  const bool has_thr = a[14] != Py_None;
  const double thr = has_thr ? real(a[14]) : 0.0, theta = real(a[15]);
  const Tensor &ws = tensor(a[16]), err = optional_tensor(a[17]);
  if (ks.dim() != 5 || vs.sizes() != ks.sizes() || !ks.is_contiguous() || !vs.is_contiguous())
    value_error("k_slab/v_slab must be contiguous (L, 1, H, N, D)");
  const int64_t L = ks.size(0), H = ks.size(2), N = ks.size(3), D = ks.size(4);
  if (!(0 <= begin && begin <= end && end <= L) || (begin <= layer && layer < end))
    value_error("gather layers (" + std::to_string(begin) + ", " + std::to_string(end) + ") must lie in [0, " +
                std::to_string(L) + ") and exclude layer " + std::to_string(layer));
  if (layer < -L || layer >= L) throw PyFailure{PyExc_IndexError, "layer out of range"};
  same_device(ks, vs, tab, segs, k, v, flags, local, spans, ws);
  k = rows_view(k);
  v = rows_view(v);
  if (ks.scalar_type() != k.scalar_type() || vs.scalar_type() != k.scalar_type() || v.scalar_type() != k.scalar_type())
    type_error("fresh and cached K/V must share a dtype");
  if (k.dim() != 4 || k.size(1) != H || k.size(3) != D || v.sizes() != k.sizes())
    value_error("fresh k/v shape " + shape_of(k) + " does not match cache " + shape_of(ks));
  if (flags.scalar_type() != at::kByte || local.scalar_type() != at::kInt || flags.numel() != N || local.numel() != N)
    value_error("flags must be uint8 (N,) and local int32 (N,)");
  if (!flags.is_contiguous() || !local.is_contiguous()) value_error("flags and local must be contiguous");
  if (tab.scalar_type() != at::kLong || tab.numel() % (2 * L)) value_error("src_tab must be int64 with 2 addresses per (chunk, layer)");
  if (segs.scalar_type() != at::kInt || segs.numel() < 6 * n_segs) value_error("segments must be int32 with 6 fields per segment");
  if (spans.scalar_type() != at::kInt || spans.numel() % 4) value_error("spans must be int32 (C, 4)");
  if ((int64_t)(ws.numel() * ws.element_size()) < CKV_LAYER1_REPAIR_WORKSPACE_BYTES || !ws.is_contiguous())
    value_error("workspace must come from layer1_repair_workspace()");
  const int64_t C = spans.numel() / 4;
  auto of = [&](at::ScalarType t, int64_t n) { return at::empty({n}, ks.options().dtype(t)); };
  Tensor dn[2], out[6];
  auto given = [](PyObject* o, Tensor* to, Py_ssize_t n) {
    if (!PyTuple_Check(o) || PyTuple_GET_SIZE(o) != n) type_error("expected a tuple of " + std::to_string(n) + " tensors");
    for (Py_ssize_t i = 0; i < n; ++i) to[i] = tensor(PyTuple_GET_ITEM(o, i));
  };
  if (a[19] != Py_None) given(a[19], dn, 2);
  else for (Tensor& t : dn) t = of(at::kFloat, N);
  if (a[18] != Py_None) {
    given(a[18], out, 6);
  } else {
    out[0] = of(at::kLong, N);
    out[1] = of(at::kLong, N);
    out[2] = of(at::kInt, N);
    out[3] = of(at::kFloat, C);
    out[4] = of(at::kByte, C);
    out[5] = of(at::kInt, CKV_COUNT_N);
  }
  const int code = dtype_code(ks);
  check(unlocked([&] {
          return ckv_layer1_repair_gather(
              ptr(ks), ptr(vs), H * N * D, N * D, (const uint64_t*)ptr(tab), int32(tab.numel() / (2 * L)), int32(L),
              int32(layer), int32(begin), int32(end), (const ckv_segment*)ptr(segs), int32(n_segs), int32(max_seg),
              ptr(k), k.stride(1), k.stride(2), ptr(v), v.stride(1), v.stride(2), int32(k.size(2)),
              (const uint8_t*)ptr(flags), (const int32_t*)ptr(local), int32(N), int32(H), int32(D), code, theta,
              (const ckv_chunk_span*)ptr(spans), int32(C), has_thr, thr, (float*)ptr(dn[0]), (float*)ptr(dn[1]),
              (int64_t*)ptr(out[0]), (int64_t*)ptr(out[1]), (int32_t*)ptr(out[2]), (float*)ptr(out[3]),
              (uint8_t*)ptr(out[4]), (int32_t*)ptr(out[5]), ptr(ws), (int64_t)(ws.numel() * ws.element_size()),
              (int32_t*)ptr(err), stream_of(ks));
        }),
        "ckv_layer1_repair_gather");
  PyObject* r = PyTuple_New(8);
  if (r == nullptr) return nullptr;
  for (int i = 0; i < 8; ++i) PyTuple_SET_ITEM(r, i, THPVariable_Wrap(i < 2 ? dn[i] : out[i - 2]));
  return r;
  CKV_PY_END
}

// extract_chunks(k_slab, v_slab, spans, err): a list of one (2, L, 1, H, end - start, D) tensor per span
PyObject* extract_chunks(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  CKV_PY_BEGIN
  need_args(n_args, 4);
  const Tensor &ks = tensor(a[0]), &vs = tensor(a[1]), err = optional_tensor(a[3]);
  same_device(ks, vs);
  if (!ks.is_contiguous() || !vs.is_contiguous() || ks.sizes() != vs.sizes())
    value_error("K/V slabs must be contiguous and of equal shape");
  need_dims(ks, 5, "K/V slabs");
  const int64_t L = ks.size(0), H = ks.size(2), N = ks.size(3), D = ks.size(4);
  // (start, end) pairs as any iterables of integers
  std::vector<std::pair<int64_t, int64_t>> spans;
  {
    THPObjectPtr seq(PySequence_Fast(a[2], "spans must be a sequence of (start, end) pairs"));
    if (!seq) throw python_error();
    auto whole = [](PyObject* o) {
      THPObjectPtr i(PyNumber_Long(o));
      if (!i) throw python_error();
      return integer(i.get());
    };
    for (Py_ssize_t i = 0; i < PySequence_Fast_GET_SIZE(seq.get()); ++i) {
      THPObjectPtr pair(PySequence_Fast(PySequence_Fast_GET_ITEM(seq.get(), i), "a span is a (start, end) pair"));
      if (!pair) throw python_error();
      if (PySequence_Fast_GET_SIZE(pair.get()) != 2) value_error("a span is a (start, end) pair");
      const int64_t start = whole(PySequence_Fast_GET_ITEM(pair.get(), 0)), end = whole(PySequence_Fast_GET_ITEM(pair.get(), 1));
      if (!(0 <= start && start <= end && end <= N))
        value_error("span [" + std::to_string(start) + ", " + std::to_string(end) + ") outside the request of " +
                    std::to_string(N) + " tokens");
      spans.emplace_back(start, end);
    }
  }
  std::vector<Tensor> bufs;
  int64_t live = 0, most = 0;
  for (const auto& [start, end] : spans) {
    bufs.push_back(at::empty({2, L, 1, H, end - start, D}, ks.options()));
    live += end > start;
    most = std::max(most, end - start);
  }
  const int code = live > 0 ? dtype_code(ks) : 0;
  // Up to 64 segments go by value with the launch; a longer list goes through device memory.
  if (live > 0 && live <= 64) {
    uint64_t dst[64];
    int32_t rows[128];
    int32_t n = 0;
    for (size_t i = 0; i < spans.size(); ++i) {
      if (spans[i].second == spans[i].first) continue;
      dst[n] = (uint64_t)(uintptr_t)bufs[i].data_ptr();
      rows[2 * n] = (int32_t)spans[i].first;
      rows[2 * n++ + 1] = (int32_t)(spans[i].second - spans[i].first);
    }
    check(unlocked([&] {
            return ckv_extract_chunks_host(ptr(ks), ptr(vs), H * N * D, N * D, dst, rows, n, int32(L), int32(H), int32(N),
                                           int32(D), code, stream_of(ks));
          }),
          "ckv_extract_chunks_host");
  } else if (live > 0) {
    // descriptors: an address per span, then (start, length) pairs; pinned, one async copy (torch's
    // pinned allocator keeps the host block until the copy has run)
    Tensor host = at::empty({live * 2}, at::TensorOptions().dtype(at::kLong).pinned_memory(true));
    int64_t* at64 = host.data_ptr<int64_t>();
    int32_t* at32 = reinterpret_cast<int32_t*>(at64 + live);
    for (size_t i = 0; i < spans.size(); ++i) {
      if (spans[i].second == spans[i].first) continue;
      *at64++ = (int64_t)(uintptr_t)bufs[i].data_ptr();
      *at32++ = (int32_t)spans[i].first;
      *at32++ = (int32_t)(spans[i].second - spans[i].first);
    }
    const Tensor d = host.to(ks.device(), /*non_blocking=*/true);
    const uint64_t* dst = (const uint64_t*)ptr(d);
    check(unlocked([&] {
            return ckv_extract_chunks(ptr(ks), ptr(vs), H * N * D, N * D, dst, (const int32_t*)(dst + live),
                                      int32(live), int32(most), int32(L), int32(H), int32(N), int32(D), code,
                                      (int32_t*)ptr(err), stream_of(ks));
          }),
          "ckv_extract_chunks");
  }
  THPObjectPtr list(PyList_New((Py_ssize_t)bufs.size()));
  if (!list) return nullptr;
  for (size_t i = 0; i < bufs.size(); ++i) PyList_SET_ITEM(list.get(), (Py_ssize_t)i, THPVariable_Wrap(bufs[i]));
  return list.release();
  CKV_PY_END
}

PyMethodDef kMethods[] = {
    {"attention_active", (PyCFunction)(void (*)(void))attention_active, METH_FASTCALL, nullptr},
    {"rope_qkv", (PyCFunction)(void (*)(void))rope_qkv, METH_FASTCALL, nullptr},
    {"add_rmsnorm", (PyCFunction)(void (*)(void))add_rmsnorm, METH_FASTCALL, nullptr},
    {"silu_mul", (PyCFunction)(void (*)(void))silu_mul, METH_FASTCALL, nullptr},
    {"linear", (PyCFunction)(void (*)(void))linear, METH_FASTCALL, nullptr},
    {"layer1_repair_gather", (PyCFunction)(void (*)(void))layer1_repair_gather, METH_FASTCALL, nullptr},
    {"extract_chunks", (PyCFunction)(void (*)(void))extract_chunks, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_torch_ops", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__torch_ops() { return PyModule_Create(&kModule); }
