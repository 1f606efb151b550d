// The operators' plain calls in native code.
//
// A decode-sized operator spends less time on the GPU (5-15 us) than its
// Python shim spent on the host (14-21 us: some forty tensor attribute reads,
// ctypes conversions, environment reads, allocations).  These functions take
// the same tensors, check that a call is plain -- exact tensors (or
// parameters) of the expected types, shapes, layout and alignment on the
// current device, no dispatch or function mode, no functorch wrapper, default
// switches -- and make the library call.  Anything else returns None, and the
// Python operator then runs its general path, which alone raises the argument
// errors, converts, copies and handles the other switches.  Nothing is kept
// between calls.
//
// Calls back to back, Python shim -> this: linear, 1 token, K=2048 N=5120 13.8
// -> 4.6 us (now its kernel's time), MoE layer, 1 token, E=128 top-8 20.7 ->
// 12.9, AITER entry with its routing, small experts 35.2 -> 16.5.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdlib>
#include <cstring>
#include <type_traits>
#include <utility>

#include "mxfp4_gfx950.h"

#ifndef MXFP4_TORCH
#error "MXFP4_TORCH: the torch build compiled against (build.py sets it)"
#endif

namespace {

struct Library {
  decltype(&mxfp4_linear_w4a16_pre) linear = nullptr;
  decltype(&mxfp4_linear_w4a16_workspace_size) linear_ws = nullptr;
  decltype(&mxfp4_moe_layer_pre) layer = nullptr;
  decltype(&mxfp4_moe_layer_workspace_size) layer_ws = nullptr;
  decltype(&mxfp4_fused_moe_pre) fused = nullptr;
  decltype(&mxfp4_fused_moe_workspace_size) fused_ws = nullptr;
  decltype(&mxfp4_moe_gemm_pre) gemm = nullptr;
  decltype(&mxfp4_moe_align) align = nullptr;
  decltype(&mxfp4_moe_align_sizes) align_sizes = nullptr;
  decltype(&mxfp4_moe_route) route = nullptr;
  decltype(&mxfp4_quant) quant = nullptr;
  decltype(&mxfp4_linear_w4a4) w4a4 = nullptr;
} lib;
PyObject* g_check = nullptr;  // Python: raises the exception of a status
PyObject* g_pre = nullptr;    // the class PrepackedWeights
PyObject *s_nibbles, *s_scales, *s_experts, *s_rows, *s_k, *s_source;

PyObject* none() { Py_RETURN_NONE; }

// f(a...) without the GIL.  The arguments are the caller's, read while it holds
// the GIL: data_ptr() may allocate (a copy-on-write storage) and throw, and an
// exception must not pass the point where the thread state is away.
template <typename... P>
int run(int (*f)(P...), std::common_type_t<P>... a) {
  PyThreadState* state = PyEval_SaveThread();
  const int rc = f(a...);
  PyEval_RestoreThread(state);
  return rc;
}

// The status' exception, or `ok` (a new reference, dropped on an error).
PyObject* finish(int rc, PyObject* ok) {
  if (rc == MXFP4_OK) return ok;
  Py_XDECREF(ok);
  PyObject* r = PyObject_CallFunction(g_check, "i", rc);
  Py_XDECREF(r);
  if (r != nullptr) PyErr_SetString(PyExc_RuntimeError, "mxfp4_amd: unknown status");
  return nullptr;
}

int code(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return MXFP4_DT_F32;
    case at::kBFloat16: return MXFP4_DT_BF16;
    case at::kHalf: return MXFP4_DT_F16;
    case at::kByte: return MXFP4_DT_U8;
    case at::kInt: return MXFP4_DT_I32;
    case at::kLong: return MXFP4_DT_I64;
    case at::kFloat8_e4m3fn: return MXFP4_DT_F8E4M3;
    case at::kFloat8_e5m2: return MXFP4_DT_F8E5M2;
    default: return -1;
  }
}

// No mode that would see (or replace) the Python path's tensor calls.
bool plain_thread() {
  if (c10::impl::dispatch_mode_enabled() || at::impl::torch_function_mode_enabled()) return false;
  const auto in = c10::impl::tls_local_dispatch_key_set().included_;
  return !in.has(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) &&
         !in.has(c10::DispatchKey::Tracer) && !in.has(c10::DispatchKey::Functionalize);
}

// The device all tensors of a call are on: the current one.
struct Call {
  c10::DeviceIndex device = -1;
  bool ok = true;

  // A contiguous tensor of the device, or null with ok = false.
  const at::Tensor* take(PyObject* o, size_t align = 1) {
    if (!ok) return nullptr;
    if (!THPVariable_CheckTypeExact(Py_TYPE(o))) return fail();
    const at::Tensor& t = THPVariable_Unpack(o);
    static const c10::DispatchKeySet wrapped(
        {c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
         c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize,
         c10::DispatchKey::Conjugate, c10::DispatchKey::Negative, c10::DispatchKey::ZeroTensor,
         c10::DispatchKey::NestedTensor});
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided ||
        t.key_set().has_any(wrapped) || !t.has_storage() || !t.is_contiguous())
      return fail();
    if (device < 0) device = t.device().index();
    if (t.device().index() != device) return fail();
    if (align > 1 && reinterpret_cast<uintptr_t>(t.const_data_ptr()) % align) return fail();
    return &t;
  }
  const at::Tensor* fail() {
    ok = false;
    return nullptr;
  }
  bool current() const { return ok && device == c10::hip::current_device(); }
  void* stream() const { return c10::hip::getCurrentHIPStream(device).stream(); }
};

template <typename T>
T* data(const at::Tensor* t) {
  return t == nullptr ? nullptr : static_cast<T*>(t->data_ptr());
}

bool shaped(const at::Tensor* t, std::initializer_list<int64_t> s) {
  return t->sizes() == at::IntArrayRef(s.begin(), s.size());
}

at::Tensor bytes(const at::Tensor& like, int64_t n) {
  return at::empty({n}, like.options().dtype(at::kByte));
}

bool env_is(const char* name, const char* value) {
  const char* v = std::getenv(name);
  return v == nullptr || std::strcmp(v, value) == 0;
}

// A prepacked copy's arrays.  False: not a plain, current copy of (w, s).
struct Pre {
  const uint8_t* nibbles = nullptr;
  const uint16_t* scales = nullptr;

  static bool same(PyObject* source, const at::Tensor& t) {
    if (!PyTuple_CheckExact(source) || PyTuple_GET_SIZE(source) != 2) return false;
    PyObject *p = PyTuple_GET_ITEM(source, 0), *v = PyTuple_GET_ITEM(source, 1);
    if (!PyLong_CheckExact(p) || !PyLong_CheckExact(v) || t.is_inference()) return false;
    return PyLong_AsUnsignedLongLong(p) == reinterpret_cast<uintptr_t>(t.const_data_ptr()) &&
           PyLong_AsUnsignedLongLong(v) == t._version();
  }
  static bool is(PyObject* o, PyObject* name, int64_t want) {
    PyObject* v = PyObject_GetAttr(o, name);
    const bool r = v != nullptr && PyLong_CheckExact(v) && PyLong_AsLongLong(v) == want;
    Py_XDECREF(v);
    return r;
  }
  bool read(Call& c, PyObject* o, int64_t experts, int64_t rows, int64_t k, const at::Tensor& w,
            const at::Tensor& s) {
    if (o == Py_None) return true;
    // nothing that only has its attributes: the general path refuses that
    if (reinterpret_cast<PyObject*>(Py_TYPE(o)) != g_pre) return false;
    bool good = is(o, s_experts, experts) && is(o, s_rows, rows) && is(o, s_k, k);
    PyObject* src = good ? PyObject_GetAttr(o, s_source) : nullptr;
    PyObject* n = src != nullptr ? PyObject_GetAttr(o, s_nibbles) : nullptr;
    PyObject* q = n != nullptr ? PyObject_GetAttr(o, s_scales) : nullptr;
    good = q != nullptr && PyTuple_CheckExact(src) && PyTuple_GET_SIZE(src) == 2 &&
           same(PyTuple_GET_ITEM(src, 0), w) && same(PyTuple_GET_ITEM(src, 1), s);
    if (good) {
      const at::Tensor *nt = c.take(n), *qt = c.take(q);
      good = c.ok;
      if (good) {
        nibbles = data<uint8_t>(nt);
        scales = data<uint16_t>(qt);
      }
    }
    Py_XDECREF(src);
    Py_XDECREF(n);
    Py_XDECREF(q);
    if (PyErr_Occurred()) PyErr_Clear();  // the general path reports it
    return good;
  }
};

bool half_type(at::ScalarType t) { return t == at::kBFloat16 || t == at::kHalf; }

// linear(x, packed, block_scales, bias, prepacked) -> Tensor or None
PyObject* linear(PyObject*, PyObject* const* a, Py_ssize_t) {
  HANDLE_TH_ERRORS
  if (!plain_thread() || !env_is("MXFP4_GFX936_BACKEND", "safe")) return none();
  Call c;
  const at::Tensor *x = c.take(a[0], 16), *w = c.take(a[1], 16), *s = c.take(a[2]);
  const at::Tensor* b = a[3] == Py_None ? nullptr : c.take(a[3]);
  if (!c.current() || !half_type(x->scalar_type()) || w->scalar_type() != at::kByte ||
      s->scalar_type() != at::kByte || w->dim() != 2 || s->dim() != 2 || x->dim() < 1)
    return none();
  const int64_t n = w->size(0), k = w->size(1) * 2;
  if (k % 128 || x->size(-1) != k || !shaped(s, {n, k / 32}) || x->numel() == 0 || n == 0)
    return none();
  if (b && (b->scalar_type() != x->scalar_type() || !shaped(b, {n}))) return none();
  Pre pre;
  if (!pre.read(c, a[4], 1, n, k, *w, *s)) return none();
  const int64_t m = x->numel() / k;
  int64_t ws_bytes = 0;
  int rc = lib.linear_ws(m, k, n, &ws_bytes);
  if (rc) return finish(rc, nullptr);
  c10::SmallVector<int64_t, 4> shape(x->sizes().begin(), x->sizes().end());
  shape.back() = n;
  at::Tensor out = at::empty(shape, x->options()), ws;
  if (ws_bytes) ws = bytes(*x, ws_bytes);
  rc = run(lib.linear, x->data_ptr(), code(x->scalar_type()), m, k, k, data<uint8_t>(w),
           data<uint8_t>(s), pre.nibbles, pre.scales, n, b ? b->data_ptr() : nullptr,
           out.data_ptr(), ws_bytes ? ws.data_ptr() : nullptr, ws_bytes, c.stream());
  return finish(rc, rc ? nullptr : THPVariable_Wrap(std::move(out)));
  END_HANDLE_TH_ERRORS
}

bool ids_type(const at::Tensor* t) {
  return t->scalar_type() == at::kInt || t->scalar_type() == at::kLong;
}

// moe_layer(x, w13, s13, w2, s2, topk_weights, topk_ids, pre13, pre2) -> Tensor or None
PyObject* moe_layer(PyObject*, PyObject* const* a, Py_ssize_t) {
  HANDLE_TH_ERRORS
  if (!plain_thread()) return none();
  Call c;
  const at::Tensor *x = c.take(a[0], 16), *w13 = c.take(a[1], 16), *s13 = c.take(a[2]),
                   *w2 = c.take(a[3], 16), *s2 = c.take(a[4]), *tw = c.take(a[5]),
                   *ids = c.take(a[6]);
  if (!c.current() || !half_type(x->scalar_type()) || x->dim() != 2 || w13->dim() != 3) return none();
  for (const at::Tensor* t : {w13, s13, w2, s2})
    if (t->scalar_type() != at::kByte) return none();
  const int64_t m = x->size(0), hidden = x->size(1), e = w13->size(0), inter = w13->size(1) / 2;
  if (m == 0 || hidden % 32 || inter % 32 || !shaped(w13, {e, 2 * inter, hidden / 2}) ||
      !shaped(s13, {e, 2 * inter, hidden / 32}) || !shaped(w2, {e, hidden, inter / 2}) ||
      !shaped(s2, {e, hidden, inter / 32}))
    return none();
  if (tw->scalar_type() != at::kFloat || !ids_type(ids) || ids->dim() != 2 || ids->size(0) != m ||
      ids->sizes() != tw->sizes())
    return none();
  Pre p13, p2;
  if (!p13.read(c, a[7], e, 2 * inter, hidden, *w13, *s13) ||
      !p2.read(c, a[8], e, hidden, inter, *w2, *s2))
    return none();
  const int top_k = (int)ids->size(1);
  int64_t ws_bytes = 0;
  int rc = lib.layer_ws(m, top_k, (int)e, hidden, inter, &ws_bytes);
  if (rc) return finish(rc, nullptr);
  at::Tensor out = at::empty({m, hidden}, x->options()), ws = bytes(*x, ws_bytes);
  rc = run(lib.layer, x->data_ptr(), code(x->scalar_type()), m, hidden, data<uint8_t>(w13),
           data<uint8_t>(s13), p13.nibbles, p13.scales, data<uint8_t>(w2), data<uint8_t>(s2),
           p2.nibbles, p2.scales, (int)e, inter, data<float>(tw), ids->data_ptr(),
           code(ids->scalar_type()), top_k, out.data_ptr(), ws.data_ptr(), ws_bytes, c.stream());
  return finish(rc, rc ? nullptr : THPVariable_Wrap(std::move(out)));
  END_HANDLE_TH_ERRORS
}

// A Python int as int64; anything else, or one out of range, is -1.
int64_t whole(PyObject* o) {
  if (!PyLong_CheckExact(o)) return -1;
  int overflow = 0;
  const long long v = PyLong_AsLongLongAndOverflow(o, &overflow);
  return overflow ? -1 : (int64_t)v;
}

// The operands both routed operators share: A (packed with A_mx, FP8 with or
// without, or a type the kernels take as it is for C), B, C, scales, routes.
struct Routed {
  const at::Tensor *A, *B, *C, *as, *bs, *amx, *bmx, *tw, *ids;
  int64_t m, e, n, k;
  int top_k;

  bool read(Call& c, PyObject* const* a, int64_t top, bool fp8) {
    A = c.take(a[0], 16), B = c.take(a[1], 16), C = c.take(a[2], 16);
    as = c.take(a[3]), bs = c.take(a[4]);
    amx = a[5] == Py_None ? nullptr : c.take(a[5]);
    bmx = c.take(a[6]), tw = c.take(a[7]), ids = c.take(a[8]);
    if (!c.current()) return false;
    if (A->dim() != 2 || B->dim() != 3 || C->dim() != 3 || ids->dim() != 2) return false;
    e = B->size(0), n = B->size(1), k = B->size(2) * 2, m = ids->size(0);
    top_k = (int)top;
    const at::ScalarType at = A->scalar_type(), ct = C->scalar_type();
    if (B->scalar_type() != at::kByte || bmx->scalar_type() != at::kByte || k % 32 || k == 0 ||
        !shaped(bmx, {e, n, k / 32}) || top < 1 || !shaped(C, {m, top, n}) ||
        !shaped(ids, {m, top}) || ids->sizes() != tw->sizes() || A->size(0) < m ||
        C->numel() == 0)
      return false;
    if (!half_type(ct) && ct != at::kFloat) return false;
    if (as->scalar_type() != at::kFloat || as->numel() < 1 || bs->scalar_type() != at::kFloat ||
        bs->numel() < e || e < 1 || top > 0x7FFFFFFF || tw->scalar_type() != at::kFloat || !ids_type(ids))
      return false;
    if (at == at::kByte) {
      return amx && amx->scalar_type() == at::kByte && A->size(1) * 2 == k &&
             shaped(amx, {A->size(0), k / 32});
    }
    if (A->size(1) != k) return false;
    if (fp8 && (at == at::kFloat8_e4m3fn || at == at::kFloat8_e5m2))
      return !amx || (amx->scalar_type() == at::kByte && shaped(amx, {A->size(0), k / 32}));
    return !amx && (at == ct || (ct == at::kFloat && half_type(at)));
  }
};

// soft(A, B, C, A_scale, B_scale, A_mx_scale, B_mx_scale, topk_weights, topk_ids,
//      mul_routed_weight, top_k) -> True or None
PyObject* soft(PyObject*, PyObject* const* a, Py_ssize_t) {
  HANDLE_TH_ERRORS
  if (!plain_thread() || !env_is("MXFP4_GFX936_BACKEND", "safe") ||
      !env_is("MXFP4_GFX950_ROUNDING", "once") || !PyBool_Check(a[9]))
    return none();
  Call c;
  Routed r;
  if (!r.read(c, a, whole(a[10]), false)) return none();
  const int act = code(r.A->scalar_type()), out = code(r.C->scalar_type());
  int64_t ws_bytes = 0;
  int rc = lib.fused_ws(r.m, r.top_k, r.e, act, out, &ws_bytes);
  if (rc) return finish(rc, nullptr);
  at::Tensor ws = bytes(*r.A, ws_bytes);
  rc = run(lib.fused, r.A->data_ptr(), act, r.A->size(0), r.A->size(1), data<uint8_t>(r.amx),
           data<uint8_t>(r.B), data<uint8_t>(r.bmx), nullptr, nullptr, r.e, r.n, r.k,
           r.C->data_ptr(), out, data<float>(r.as), data<float>(r.bs), data<float>(r.tw),
           a[9] == Py_True ? 1 : 0, r.ids->data_ptr(), code(r.ids->scalar_type()), r.m, r.top_k,
           ws.data_ptr(), ws_bytes, c.stream());
  Py_INCREF(Py_True);
  return finish(rc, Py_True);
  END_HANDLE_TH_ERRORS
}

// routed(A, B, C, A_scale, B_scale, A_mx_scale, B_mx_scale, topk_weights, topk_ids,
//        mul_routed_weight, top_k, sorted_ids, expert_ids, num_post_padded, block_m)
//        -> True or None
PyObject* routed(PyObject*, PyObject* const* a, Py_ssize_t) {
  HANDLE_TH_ERRORS
  if (!plain_thread() || !PyBool_Check(a[9])) return none();
  Call c;
  Routed r;
  if (!r.read(c, a, whole(a[10]), true)) return none();
  const at::Tensor *srt = c.take(a[11]), *exp = c.take(a[12]), *npp = c.take(a[13]);
  const int64_t bm = whole(a[14]);
  if (!c.ok || srt->scalar_type() != at::kInt || exp->scalar_type() != at::kInt ||
      npp->scalar_type() != at::kInt || npp->numel() != 1 ||
      // asserted by the general path, also of a dimension of size 1
      r.tw->stride(1) != 1 || srt->dim() != 1 || srt->stride(0) != 1 || bm < 16 || bm % 16 ||
      bm > 0x7FFFFFFF || srt->numel() == 0 || srt->numel() % bm ||
      exp->numel() * bm < srt->numel())
    return none();
  const int rc = run(lib.gemm, r.A->data_ptr(), code(r.A->scalar_type()), r.A->size(0),
                     r.A->size(1), data<uint8_t>(r.amx), data<uint8_t>(r.B), data<uint8_t>(r.bmx),
                     nullptr, nullptr, r.e, r.n, r.k, r.C->data_ptr(), code(r.C->scalar_type()),
                     r.n, data<float>(r.as), data<float>(r.bs), data<float>(r.tw),
                     a[9] == Py_True ? 1 : 0, data<int32_t>(srt), data<int32_t>(exp),
                     data<int32_t>(npp), srt->numel(), (int)bm, r.ids->numel(), r.top_k,
                     c.stream());
  Py_INCREF(Py_True);
  return finish(rc, Py_True);
  END_HANDLE_TH_ERRORS
}

// align(topk_ids, num_experts, block_m) -> (sorted_ids, expert_ids, num_post_padded) or None
PyObject* align(PyObject*, PyObject* const* a, Py_ssize_t) {
  HANDLE_TH_ERRORS
  if (!plain_thread()) return none();
  Call c;
  const at::Tensor* ids = c.take(a[0]);
  if (!c.current() || !ids_type(ids)) return none();
  const int64_t e = whole(a[1]), bm = whole(a[2]);
  if (e < 1 || e > 0x7FFFFFFF || bm < 1 || bm > 0x7FFFFFFF) return none();
  const int64_t n = ids->numel();
  int64_t ms = 0, mb = 0, wsb = 0;
  int rc = lib.align_sizes(n, (int)e, (int)bm, &ms, &mb, &wsb);
  if (rc) return finish(rc, nullptr);
  const auto opt = ids->options().dtype(at::kInt);
  at::Tensor sorted = at::empty({ms}, opt), experts = at::empty({mb}, opt),
             npp = at::empty({1}, opt), ws = bytes(*ids, wsb > 4 ? wsb : 4);
  rc = run(lib.align, ids->data_ptr(), code(ids->scalar_type()), n, (int)e, (int)bm,
           data<int32_t>(&sorted), data<int32_t>(&experts), data<int32_t>(&npp), ws.data_ptr(), wsb,
           c.stream());
  if (rc) return finish(rc, nullptr);
  return Py_BuildValue("(NNN)", THPVariable_Wrap(std::move(sorted)),
                       THPVariable_Wrap(std::move(experts)), THPVariable_Wrap(std::move(npp)));
  END_HANDLE_TH_ERRORS
}

// route_topk(logits, top_k, renormalize, int32 ids) -> (weights, ids) or None
PyObject* route_topk(PyObject*, PyObject* const* a, Py_ssize_t) {
  HANDLE_TH_ERRORS
  if (!plain_thread()) return none();
  Call c;
  const at::Tensor* l = c.take(a[0]);
  if (!c.current() || l->scalar_type() != at::kFloat || l->dim() < 1 || l->numel() == 0)
    return none();
  const int64_t e = l->size(-1);
  const int64_t top = whole(a[1]);
  if (top < 1 || top > e || top > 64 || e > 1024) return none();
  const auto type = PyObject_IsTrue(a[3]) ? at::kInt : at::kLong;
  c10::SmallVector<int64_t, 4> shape(l->sizes().begin(), l->sizes().end());
  shape.back() = top;
  at::Tensor w = at::empty(shape, l->options()), ids = at::empty(shape, l->options().dtype(type));
  const int renorm = PyObject_IsTrue(a[2]) ? 1 : 0;
  const int rc = run(lib.route, data<float>(l), l->numel() / e, (int)e, e, (int)top, renorm,
                     data<float>(&w), ids.data_ptr(), code(type), c.stream());
  if (rc) return finish(rc, nullptr);
  return Py_BuildValue("(NN)", THPVariable_Wrap(std::move(w)), THPVariable_Wrap(std::move(ids)));
  END_HANDLE_TH_ERRORS
}

// quant(x, mode) -> (packed, scales) or None
PyObject* quant(PyObject*, PyObject* const* a, Py_ssize_t) {
  HANDLE_TH_ERRORS
  if (!plain_thread()) return none();
  Call c;
  const at::Tensor* x = c.take(a[0]);
  const int mode = (int)whole(a[1]);
  if (!c.current() || mode < 0 || x->dim() < 1 || x->numel() == 0 || x->size(-1) % 32 ||
      !(half_type(x->scalar_type()) || x->scalar_type() == at::kFloat))
    return none();
  const int64_t k = x->size(-1);
  c10::SmallVector<int64_t, 4> shape(x->sizes().begin(), x->sizes().end());
  const auto opt = x->options().dtype(at::kByte);
  shape.back() = k / 2;
  at::Tensor packed = at::empty(shape, opt);
  shape.back() = k / 32;
  at::Tensor scales = at::empty(shape, opt);
  const int rc = run(lib.quant, x->data_ptr(), code(x->scalar_type()), x->numel() / k, k, k, mode,
                     data<uint8_t>(&packed), data<uint8_t>(&scales), c.stream());
  if (rc) return finish(rc, nullptr);
  return Py_BuildValue("(NN)", THPVariable_Wrap(std::move(packed)),
                       THPVariable_Wrap(std::move(scales)));
  END_HANDLE_TH_ERRORS
}

// w4a4(a_packed, a_scales, w_packed, w_scales, out like: bf16 0 / fp16 1 / fp32 2) -> Tensor or None
PyObject* w4a4(PyObject*, PyObject* const* a, Py_ssize_t) {
  HANDLE_TH_ERRORS
  if (!plain_thread()) return none();
  Call c;
  const at::Tensor *x = c.take(a[0], 16), *xs = c.take(a[1]), *w = c.take(a[2], 16),
                   *ws = c.take(a[3]);
  if (!c.current() || x->dim() != 2 || w->dim() != 2) return none();
  for (const at::Tensor* t : {x, xs, w, ws})
    if (t->scalar_type() != at::kByte) return none();
  const int64_t m = x->size(0), n = w->size(0), k = x->size(1) * 2;
  if (w->size(1) * 2 != k || k % 32 || k == 0 || m == 0 || n == 0 || !shaped(xs, {m, k / 32}) ||
      !shaped(ws, {n, k / 32}))
    return none();
  const int64_t t = whole(a[4]);
  if (t < 0 || t > 2) return none();
  const auto type = t == 0 ? at::kBFloat16 : (t == 1 ? at::kHalf : at::kFloat);
  at::Tensor out = at::empty({m, n}, x->options().dtype(type));
  const int rc = run(lib.w4a4, data<uint8_t>(x), data<uint8_t>(xs), m, k, data<uint8_t>(w),
                     data<uint8_t>(ws), n, out.data_ptr(), code(type), c.stream());
  return finish(rc, rc ? nullptr : THPVariable_Wrap(std::move(out)));
  END_HANDLE_TH_ERRORS
}

// bind(check, PrepackedWeights, address, ...): the library's entry points, in Library's order
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
  constexpr Py_ssize_t kEntries = sizeof(Library) / sizeof(void*);
  if (n != 2 + kEntries) {
    PyErr_SetString(PyExc_TypeError, "bind: wrong number of entry points");
    return nullptr;
  }
  void* at[kEntries];
  for (Py_ssize_t i = 0; i < kEntries; ++i) {
    at[i] = PyLong_AsVoidPtr(a[2 + i]);
    if (at[i] == nullptr) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "bind: null entry point");
      return nullptr;
    }
  }
  std::memcpy(static_cast<void*>(&lib), at, sizeof(lib));
  for (Py_ssize_t i = 0; i < 2; ++i) Py_INCREF(a[i]);
  Py_XDECREF(std::exchange(g_check, a[0]));
  Py_XDECREF(std::exchange(g_pre, a[1]));
  Py_RETURN_NONE;
}

// Fixed argument counts: a wrong one is refused here, not read past.
template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t), int N>
PyObject* counted(PyObject* self, PyObject* const* a, Py_ssize_t n) {
  if (n != N || lib.linear == nullptr) {
    PyErr_Format(PyExc_TypeError, "expected %d arguments (after bind), got %zd", N, n);
    return nullptr;
  }
  return F(self, a, n);
}

#define ENTRY(name, n) \
  {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(&counted<name, n>)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    ENTRY(linear, 5), ENTRY(moe_layer, 9), ENTRY(soft, 11), ENTRY(routed, 15), ENTRY(align, 3),
    ENTRY(route_topk, 4), ENTRY(quant, 2), ENTRY(w4a4, 5),
    {"bind", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(&bind)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) {
  s_nibbles = PyUnicode_InternFromString("nibbles");
  s_scales = PyUnicode_InternFromString("scales");
  s_experts = PyUnicode_InternFromString("experts");
  s_rows = PyUnicode_InternFromString("rows");
  s_k = PyUnicode_InternFromString("k");
  s_source = PyUnicode_InternFromString("source");
  PyObject* m = PyModule_Create(&module);
  // at::Tensor is read through inlined accessors: right for this torch only
  if (m != nullptr && PyModule_AddStringConstant(m, "TORCH", MXFP4_TORCH) != 0) Py_CLEAR(m);
  return m;
}
