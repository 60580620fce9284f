// Host side of the operators as one CPython extension (testt_amd/_soupk_host.so): the C ABI's entry
// points with typed argument conversion, and the operators' checks, allocations and launch in one
// native call each.
//
// Reason: a training program's small calls are bound by the host.  Through ctypes an entry point of
// 16 arguments costs about 2 us more than its launch, and the checks and torch.empty calls around it
// 10 - 20 us of Python.  Eager forward + backward on MI355X, before and after (us): add + RMSNorm of 300
// rows 49 / 36, q|k|v projection of 16 rows 71 / 51 (its first pass on new weights, whose launch
// arguments are made then, 189 / 181), RoPE + attention of rows of 512 to 128 tokens 67 / 49, the
// padded form 122 / 95.  A GEMM takes its native call only while no tuned table is loaded.
//
// An operator here takes only the common case -- plain tensors of the expected types, contiguous, on
// one device, with matching shapes -- and returns None for anything else; the Python caller then
// runs its own checks, which convert or raise as they always did.  Nothing is cached, no state is
// shared between threads beyond the table of entry points (filled once, under the import of the
// library), and the GIL is released around every entry point, as ctypes releases it.

#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <cstring>
#include <tuple>
#include <type_traits>
#include <utility>

#include "../../include/soupk.h"

namespace {

using at::Tensor;

// ---- entry points ------------------------------------------------------------------------------

#define SOUPK_ENTRIES(X)                                                                          \
  X(soupk_nf4_unpack) X(soupk_nf4_unpack_multi) X(soupk_nf4_unpack_multi_lora)                    \
  X(soupk_index_inverse) X(soupk_sum_partials) X(soupk_rmsnorm_fwd) X(soupk_rmsnorm_bwd)          \
  X(soupk_rope_pack_fwd) X(soupk_rope_pack_bwd) X(soupk_rope_pack_tokens) X(soupk_swiglu_fwd)     \
  X(soupk_swiglu_bwd_inplace) X(soupk_head_stats_grad) X(soupk_head_stats_grad_rows)              \
  X(soupk_head_plan) X(soupk_head_stats_grad_planned) X(soupk_head_finish) X(soupk_head_dh)       \
  X(soupk_attention_fwd) X(soupk_attention_bwd) X(soupk_attention_varlen_fwd)                     \
  X(soupk_attention_varlen_bwd) X(soupk_lora_stage) X(soupk_lora_fwd) X(soupk_lora_rope_fwd)      \
  X(soupk_lora_bwd_rows) X(soupk_lora_bwd_params) X(soupk_lora_bwd_params_noalloc)                \
  X(soupk_gemm_tn) X(soupk_gemm_nn_nf4) X(soupk_gemm_tn_nf4) X(soupk_gemm_tn_nf4_split)           \
  X(soupk_gemm_nn_nf4_split) X(soupk_gemm_lt) X(soupk_gemm_nn) X(soupk_gemm_nn_workspace)         \
  X(soupk_layer_fwd) X(soupk_layer_bwd)

#define X(name) decltype(&name) p_##name = nullptr;
SOUPK_ENTRIES(X)
#undef X

template <class T>
T arg(PyObject* o) {
  if constexpr (std::is_floating_point_v<T>) {
    return static_cast<T>(PyFloat_AsDouble(o));
  } else if constexpr (std::is_pointer_v<T>) {
    if (o == Py_None) return nullptr;
    if (PyLong_Check(o))
      return reinterpret_cast<T>(static_cast<uintptr_t>(PyLong_AsUnsignedLongLongMask(o)));
    PyErr_SetString(PyExc_TypeError, "an address (int) or None is expected");
    return nullptr;
  } else {
    return static_cast<T>(PyLong_AsUnsignedLongLongMask(o));
  }
}

template <class... A, std::size_t... I>
PyObject* invoke(int (*fn)(A...), PyObject* const* a, Py_ssize_t n, std::index_sequence<I...>) {
  if (n != static_cast<Py_ssize_t>(sizeof...(A)))
    return PyErr_Format(PyExc_TypeError, "%d arguments are expected, got %zd",
                        static_cast<int>(sizeof...(A)), n);
  if (fn == nullptr) return PyErr_Format(PyExc_RuntimeError, "the soupk library is not bound");
  const std::tuple<A...> args{arg<A>(a[I])...};
  if (PyErr_Occurred()) return nullptr;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = fn(std::get<I>(args)...);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
}

template <class... A>
PyObject* invoke(int (*fn)(A...), PyObject* const* a, Py_ssize_t n) {
  return invoke(fn, a, n, std::index_sequence_for<A...>{});
}

#define X(name)                                                               \
  PyObject* call_##name(PyObject*, PyObject* const* a, Py_ssize_t n) {        \
    return invoke(p_##name, a, n);                                            \
  }
SOUPK_ENTRIES(X)
#undef X

// bind(name, address): the entry point's address in the loaded library; True when known here.
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 2) return PyErr_Format(PyExc_TypeError, "bind(name, address)");
  const char* name = PyUnicode_AsUTF8(a[0]);
  const auto addr = static_cast<uintptr_t>(PyLong_AsUnsignedLongLongMask(a[1]));
  if (name == nullptr || PyErr_Occurred()) return nullptr;
#define X(e)                                   \
  if (!std::strcmp(name, #e)) {                \
    p_##e = reinterpret_cast<decltype(p_##e)>(addr); \
    Py_RETURN_TRUE;                            \
  }
  SOUPK_ENTRIES(X)
#undef X
  Py_RETURN_FALSE;
}

// ---- operators ---------------------------------------------------------------------------------

// The tensor behind a plain torch.Tensor or Parameter (no subclass: those keep the Python path).
const Tensor* plain(PyObject* o) {
  return THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr;
}

// An optional tensor argument: false when it is something else than None or a plain tensor.
bool optional(PyObject* o, const Tensor*& t) {
  t = nullptr;
  if (o == Py_None) return true;
  t = plain(o);
  return t != nullptr;
}

bool is(const Tensor& t, at::ScalarType dt, int64_t dims, const at::Device& dev) {
  return t.scalar_type() == dt && t.dim() == dims && t.is_cuda() && t.device() == dev &&
         t.layout() == at::kStrided && t.is_contiguous();
}

bool shape2(const Tensor& t, int64_t r, int64_t c) { return t.size(0) == r && t.size(1) == c; }

void* ptr(const Tensor* t) { return t == nullptr ? nullptr : t->data_ptr(); }
template <class T>
T* ptr(const Tensor* t) {
  return static_cast<T*>(ptr(t));
}
template <class T>
T* ptr(const Tensor& t) {
  return static_cast<T*>(t.data_ptr());
}

void* stream_of(const Tensor& t) {
  return c10::hip::getCurrentHIPStream(t.device().index()).stream();
}

Tensor empty(at::IntArrayRef size, at::ScalarType dt, const at::Device& dev) {
  return at::empty(size, at::TensorOptions().dtype(dt).device(dev));
}

PyObject* g_error = nullptr;        // testt_amd._ext.SoupkError
const char* (*p_status_string)(int) = nullptr;

// The GIL given up for a scope, taken back also when an exception leaves it: a tensor without a
// storage (a functorch wrapper, for one) throws from data_ptr, and HANDLE_TH_ERRORS sets the Python
// error from it.
class NoGil {
 public:
  NoGil() : state_(PyEval_SaveThread()) {}
  ~NoGil() { PyEval_RestoreThread(state_); }
  NoGil(const NoGil&) = delete;
  NoGil& operator=(const NoGil&) = delete;

 private:
  PyThreadState* state_;
};

// The launch's status as the Python layer reports it; true when it succeeded.
template <class F>
bool launched(const char* name, F&& f) {
  const int rc = [&] {
    const NoGil released;
    return f();
  }();
  if (rc == 0) return true;
  const char* text = p_status_string ? p_status_string(rc) : nullptr;
  PyErr_Format(g_error ? g_error : PyExc_RuntimeError, "%s failed with status %d: %s", name, rc,
               text ? text : "?");
  return false;
}

PyObject* pack(std::initializer_list<Tensor> ts) {
  PyObject* out = PyTuple_New(static_cast<Py_ssize_t>(ts.size()));
  Py_ssize_t i = 0;
  for (const Tensor& t : ts) {
    PyObject* o = t.defined() ? THPVariable_Wrap(t) : Py_NewRef(Py_None);
    PyTuple_SET_ITEM(out, i++, o);
  }
  return out;
}

#define OP(name) PyObject* name(PyObject*, PyObject* const* a, Py_ssize_t n)
#define ARGS(count) \
  if (n != (count)) return PyErr_Format(PyExc_TypeError, "%d arguments are expected", (count))
#define ELSE_PYTHON Py_RETURN_NONE
#define NUM(i) PyLong_AsLongLong(a[i])

// rmsnorm_fwd(x, delta, weight, eps, pad_idx, padded_rows, inv) -> (s, y, ypad, rstd)
OP(rmsnorm_fwd) {
  HANDLE_TH_ERRORS
  ARGS(7);
  const Tensor *x = plain(a[0]), *w = plain(a[2]), *delta, *pad, *inv;
  if (!x || !w || !optional(a[1], delta) || !optional(a[4], pad) || !optional(a[6], inv) ||
      x->dim() != 2)
    ELSE_PYTHON;
  const at::Device dev = x->device();
  const int64_t rows = x->size(0), H = x->size(1), padded = pad ? NUM(5) : 0;
  if (!is(*x, at::kFloat, 2, dev) || !is(*w, at::kFloat, 1, dev) || w->size(0) != H ||
      (delta && (!is(*delta, at::kHalf, 2, dev) || !shape2(*delta, rows, H))) ||
      (pad && (!is(*pad, at::kLong, 1, dev) || pad->size(0) != rows || padded < 0 ||
               (inv == nullptr && padded != rows))) ||
      (inv && (!pad || !is(*inv, at::kInt, 1, dev) || inv->size(0) != padded)) || rows == 0)
    ELSE_PYTHON;
  const double eps = PyFloat_AsDouble(a[3]);
  if (PyErr_Occurred()) return nullptr;
  Tensor s = delta ? empty({rows, H}, at::kFloat, dev) : *x;
  Tensor y = empty({rows, H}, at::kHalf, dev), rstd = empty({rows}, at::kFloat, dev);
  Tensor ypad = empty({padded, H}, at::kFloat, dev);
  void* st = stream_of(*x);
  if (!launched("soupk_rmsnorm_fwd", [&] {
        return p_soupk_rmsnorm_fwd(ptr<float>(x), ptr<uint16_t>(delta), ptr<float>(w),
                                   delta ? ptr<float>(s) : nullptr, ptr<uint16_t>(y),
                                   pad ? ptr<float>(ypad) : nullptr, ptr<int64_t>(pad),
                                   ptr<int32_t>(inv), ptr<float>(rstd), rows, padded,
                                   static_cast<int32_t>(H), static_cast<float>(eps), st);
      }))
    return nullptr;
  return pack({s, y, ypad, rstd});
  END_HANDLE_TH_ERRORS
}

// rmsnorm_bwd(s, rstd, weight, pad_idx, grad_s, grad_y, grad_ypad, want_delta) -> (dx, ddelta)
OP(rmsnorm_bwd) {
  HANDLE_TH_ERRORS
  ARGS(8);
  const Tensor *s = plain(a[0]), *rstd = plain(a[1]), *w = plain(a[2]), *pad, *gs, *gy, *gp;
  if (!s || !rstd || !w || !optional(a[3], pad) || !optional(a[4], gs) || !optional(a[5], gy) ||
      !optional(a[6], gp) || s->dim() != 2)
    ELSE_PYTHON;
  const at::Device dev = s->device();
  const int64_t rows = s->size(0), H = s->size(1);
  const bool want_delta = a[7] == Py_True;
  const bool has_pad = gp && pad && gp->numel() > 0;
  if (!is(*s, at::kFloat, 2, dev) || !is(*rstd, at::kFloat, 1, dev) || rstd->size(0) != rows ||
      !is(*w, at::kFloat, 1, dev) || w->size(0) != H ||
      (gs && (!is(*gs, at::kFloat, 2, dev) || !shape2(*gs, rows, H))) ||
      (gy && (!is(*gy, at::kHalf, 2, dev) || !shape2(*gy, rows, H))) ||
      (has_pad && (!is(*gp, at::kFloat, 2, dev) || gp->size(1) != H ||
                   !is(*pad, at::kLong, 1, dev) || pad->size(0) != rows)) ||
      rows == 0)
    ELSE_PYTHON;
  Tensor dx = empty({rows, H}, at::kFloat, dev);
  Tensor ddelta = want_delta ? empty({rows, H}, at::kHalf, dev) : Tensor();
  void* st = stream_of(*s);
  if (!launched("soupk_rmsnorm_bwd", [&] {
        return p_soupk_rmsnorm_bwd(
            ptr<float>(s), ptr<float>(rstd), ptr<float>(w), ptr<uint16_t>(gy),
            has_pad ? ptr<float>(gp) : nullptr, has_pad ? ptr<int64_t>(pad) : nullptr,
            ptr<float>(gs), ptr<float>(dx), want_delta ? ptr<uint16_t>(ddelta) : nullptr, rows,
            has_pad ? gp->size(0) : 0, static_cast<int32_t>(H), st);
      }))
    return nullptr;
  return pack({dx, ddelta});
  END_HANDLE_TH_ERRORS
}

// The shared operands of the RoPE launches: qkv rows, LoRA deltas of one type, tables, positions.
struct RopeArgs {
  const Tensor *qkv, *lq, *lv, *cos, *sin, *pos;
  int64_t rows, batch, seq, nh, nkv, hd;
  int32_t code;
};

bool rope_args(PyObject* const* a, int64_t batch, int64_t seq, int64_t nh, int64_t nkv, int64_t hd,
               RopeArgs& r) {
  r.qkv = plain(a[0]);
  r.cos = plain(a[3]);
  r.sin = plain(a[4]);
  r.pos = plain(a[5]);
  if (!r.qkv || !r.cos || !r.sin || !r.pos || !optional(a[1], r.lq) || !optional(a[2], r.lv) ||
      batch < 0 || seq < 1 || nh < 1 || nkv < 1 || hd < 2 || hd % 2 || r.qkv->dim() != 2)
    return false;
  const at::Device dev = r.qkv->device();
  r.rows = r.qkv->size(0);
  r.batch = batch, r.seq = seq, r.nh = nh, r.nkv = nkv, r.hd = hd;
  const Tensor* first = r.lq ? r.lq : r.lv;
  const at::ScalarType lt = first ? first->scalar_type() : at::kHalf;
  r.code = lt == at::kHalf ? 0 : 1;
  auto table = [&](const Tensor& t) {
    return is(t, at::kFloat, 2, dev) && t.size(0) >= seq && t.size(1) == hd;
  };
  return is(*r.qkv, at::kHalf, 2, dev) && r.qkv->size(1) == (nh + 2 * nkv) * hd &&
         (lt == at::kHalf || lt == at::kFloat) &&
         (!r.lq || (is(*r.lq, lt, 2, dev) && shape2(*r.lq, r.rows, nh * hd))) &&
         (!r.lv || (is(*r.lv, lt, 2, dev) && shape2(*r.lv, r.rows, nkv * hd))) &&
         table(*r.cos) && table(*r.sin) && is(*r.pos, at::kLong, 1, dev) &&
         r.pos->size(0) == r.rows && r.rows > 0;
}

// rope_tokens(qkv, lq, lv, cos, sin, pos, batch, seq, nh, nkv) -> out (head dim 128)
OP(rope_tokens) {
  HANDLE_TH_ERRORS
  ARGS(10);
  RopeArgs r;
  if (!rope_args(a, NUM(6), NUM(7), NUM(8), NUM(9), 128, r) || PyErr_Occurred()) {
    PyErr_Clear();
    ELSE_PYTHON;
  }
  Tensor out = empty({r.rows, r.qkv->size(1)}, at::kHalf, r.qkv->device());
  void* st = stream_of(out);
  if (!launched("soupk_rope_pack_tokens", [&] {
        return p_soupk_rope_pack_tokens(
            ptr<uint16_t>(r.qkv), ptr(r.lq), ptr(r.lv), r.code, ptr<float>(r.cos),
            ptr<float>(r.sin), ptr<int64_t>(r.pos), ptr<uint16_t>(out), r.rows,
            static_cast<int32_t>(r.batch), static_cast<int32_t>(r.seq),
            static_cast<int32_t>(r.nh), static_cast<int32_t>(r.nkv), 128, st);
      }))
    return nullptr;
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// rope_fwd(qkv, lq, lv, cos, sin, pos, inv, batch, seq, nh, nkv, hd) -> (q, k, v)
OP(rope_fwd) {
  HANDLE_TH_ERRORS
  ARGS(12);
  RopeArgs r;
  const Tensor* inv;
  if (!optional(a[6], inv) || !rope_args(a, NUM(7), NUM(8), NUM(9), NUM(10), NUM(11), r) ||
      PyErr_Occurred()) {
    PyErr_Clear();
    ELSE_PYTHON;
  }
  const at::Device dev = r.qkv->device();
  const int64_t slots = r.batch * r.seq;
  if (inv ? !is(*inv, at::kInt, 1, dev) || inv->size(0) != slots : slots != r.rows) ELSE_PYTHON;
  Tensor q = empty({r.batch, r.nh, r.seq, r.hd}, at::kHalf, dev);
  Tensor k = empty({r.batch, r.nkv, r.seq, r.hd}, at::kHalf, dev);
  Tensor v = empty({r.batch, r.nkv, r.seq, r.hd}, at::kHalf, dev);
  void* st = stream_of(q);
  if (!launched("soupk_rope_pack_fwd", [&] {
        return p_soupk_rope_pack_fwd(
            ptr<uint16_t>(r.qkv), ptr(r.lq), ptr(r.lv), r.code, ptr<float>(r.cos),
            ptr<float>(r.sin), ptr<int64_t>(r.pos), ptr<int32_t>(inv), ptr<uint16_t>(q),
            ptr<uint16_t>(k), ptr<uint16_t>(v), r.rows, static_cast<int32_t>(r.batch),
            static_cast<int32_t>(r.seq), static_cast<int32_t>(r.nh),
            static_cast<int32_t>(r.nkv), static_cast<int32_t>(r.hd), st);
      }))
    return nullptr;
  return pack({q, k, v});
  END_HANDLE_TH_ERRORS
}

// rope_bwd(gq, gk, gv, cos, sin, pos, batch, seq, nh, nkv, hd) -> dqkv
OP(rope_bwd) {
  HANDLE_TH_ERRORS
  ARGS(11);
  const Tensor *gq = plain(a[0]), *gk = plain(a[1]), *gv = plain(a[2]), *cos = plain(a[3]),
               *sin = plain(a[4]), *pos = plain(a[5]);
  const int64_t B = NUM(6), T = NUM(7), nh = NUM(8), nkv = NUM(9), hd = NUM(10);
  if (PyErr_Occurred()) return nullptr;
  if (!gq || !gk || !gv || !cos || !sin || !pos || !pos->is_cuda()) ELSE_PYTHON;
  const at::Device dev = pos->device();
  auto grad = [&](const Tensor& t, int64_t heads) {
    return is(t, at::kHalf, 4, dev) && t.size(0) == B && t.size(1) == heads && t.size(2) == T &&
           t.size(3) == hd;
  };
  auto table = [&](const Tensor& t) {
    return is(t, at::kFloat, 2, dev) && t.size(0) >= T && t.size(1) == hd;
  };
  const int64_t rows = pos->numel();
  if (!grad(*gq, nh) || !grad(*gk, nkv) || !grad(*gv, nkv) || !table(*cos) || !table(*sin) ||
      !is(*pos, at::kLong, 1, dev) || rows == 0)
    ELSE_PYTHON;
  Tensor d = empty({rows, (nh + 2 * nkv) * hd}, at::kHalf, dev);
  void* st = stream_of(d);
  if (!launched("soupk_rope_pack_bwd", [&] {
        return p_soupk_rope_pack_bwd(ptr<uint16_t>(gq), ptr<uint16_t>(gk), ptr<uint16_t>(gv),
                                     ptr<float>(cos), ptr<float>(sin), ptr<int64_t>(pos),
                                     ptr<uint16_t>(d), rows, static_cast<int32_t>(B),
                                     static_cast<int32_t>(T), static_cast<int32_t>(nh),
                                     static_cast<int32_t>(nkv), static_cast<int32_t>(hd), st);
      }))
    return nullptr;
  return THPVariable_Wrap(d);
  END_HANDLE_TH_ERRORS
}

constexpr int64_t kHeadDim = 128;

// varlen_fwd(qkv_r, cu, nh, nkv, scale) -> (out, lse)
OP(varlen_fwd) {
  HANDLE_TH_ERRORS
  ARGS(5);
  const Tensor *q = plain(a[0]), *cu = plain(a[1]);
  const int64_t nh = NUM(2), nkv = NUM(3);
  const double scale = PyFloat_AsDouble(a[4]);
  if (PyErr_Occurred()) return nullptr;
  if (!q || !cu || q->dim() != 2 || nh < 1 || nkv < 1) ELSE_PYTHON;
  const at::Device dev = q->device();
  const int64_t M = q->size(0);
  if (!is(*q, at::kHalf, 2, dev) || q->size(1) != (nh + 2 * nkv) * kHeadDim ||
      !is(*cu, at::kInt, 1, dev) || cu->size(0) < 1)
    ELSE_PYTHON;
  Tensor out = empty({M, nh * kHeadDim}, at::kHalf, dev), lse = empty({nh, M}, at::kFloat, dev);
  void* st = stream_of(out);
  if (!launched("soupk_attention_varlen_fwd", [&] {
        return p_soupk_attention_varlen_fwd(
            ptr<uint16_t>(q), ptr<int32_t>(cu), static_cast<int32_t>(cu->size(0) - 1),
            ptr<uint16_t>(out), ptr<float>(lse), M, static_cast<int32_t>(nh),
            static_cast<int32_t>(nkv), kHeadDim, static_cast<float>(scale), st);
      }))
    return nullptr;
  return pack({out, lse});
  END_HANDLE_TH_ERRORS
}

// varlen_bwd(qkv_r, cu, out, lse, dout, scale, nh, nkv, cos, sin, pos, batch, seq) -> dqkv
OP(varlen_bwd) {
  HANDLE_TH_ERRORS
  ARGS(13);
  const Tensor *q = plain(a[0]), *cu = plain(a[1]), *out = plain(a[2]), *lse = plain(a[3]),
               *dout = plain(a[4]), *cos, *sin, *pos;
  const double scale = PyFloat_AsDouble(a[5]);
  const int64_t nh = NUM(6), nkv = NUM(7), batch = NUM(11), seq = NUM(12);
  if (PyErr_Occurred()) return nullptr;
  if (!q || !cu || !out || !lse || !dout || !optional(a[8], cos) || !optional(a[9], sin) ||
      !optional(a[10], pos) || q->dim() != 2 || nh < 1 || nkv < 1)
    ELSE_PYTHON;
  const at::Device dev = q->device();
  const int64_t M = q->size(0), HD = nh * kHeadDim;
  auto table = [&](const Tensor* t) {
    return t && is(*t, at::kFloat, 2, dev) && t->size(0) >= seq && t->size(1) == kHeadDim;
  };
  const bool rope = cos || sin || pos;
  if (!is(*q, at::kHalf, 2, dev) || q->size(1) != HD + 2 * nkv * kHeadDim ||
      !is(*cu, at::kInt, 1, dev) || cu->size(0) < 1 || !is(*out, at::kHalf, 2, dev) ||
      !shape2(*out, M, HD) || !is(*lse, at::kFloat, 2, dev) || !shape2(*lse, nh, M) ||
      !is(*dout, at::kHalf, 2, dev) || !shape2(*dout, M, HD) ||
      (rope && (!table(cos) || !table(sin) || !pos || !is(*pos, at::kLong, 1, dev) ||
                pos->size(0) != M)))
    ELSE_PYTHON;
  Tensor d = empty({M, q->size(1)}, at::kHalf, dev);
  Tensor ws = empty({(M * nh + 3) / 4 * 4 + 2 * M * HD}, at::kFloat, dev);
  void* st = stream_of(d);
  if (!launched("soupk_attention_varlen_bwd", [&] {
        return p_soupk_attention_varlen_bwd(
            ptr<uint16_t>(q), ptr<int32_t>(cu), static_cast<int32_t>(cu->size(0) - 1),
            ptr<uint16_t>(out), ptr<uint16_t>(dout), ptr<float>(lse), ptr<float>(cos),
            ptr<float>(sin), ptr<int64_t>(pos), rope ? batch * seq : 0,
            rope ? static_cast<int32_t>(seq) : 0, ptr<float>(ws), ptr<uint16_t>(d), M,
            static_cast<int32_t>(nh), static_cast<int32_t>(nkv), kHeadDim,
            static_cast<float>(scale), st);
      }))
    return nullptr;
  return THPVariable_Wrap(d);
  END_HANDLE_TH_ERRORS
}

// q [B, NH, T, 128], k and v [B, NKV, T, 128] fp16 and the optional key flags [B, T].
struct PaddedArgs {
  const Tensor *q, *k, *v, *valid;
  int64_t B, NH, T, NKV;
};

bool padded_args(PyObject* const* a, PaddedArgs& p) {
  p.q = plain(a[0]), p.k = plain(a[1]), p.v = plain(a[2]);
  if (!p.q || !p.k || !p.v || !optional(a[3], p.valid) || p.q->dim() != 4 || p.k->dim() != 4)
    return false;
  const at::Device dev = p.q->device();
  p.B = p.q->size(0), p.NH = p.q->size(1), p.T = p.q->size(2), p.NKV = p.k->size(1);
  auto heads = [&](const Tensor& t, int64_t h) {
    return is(t, at::kHalf, 4, dev) && t.size(0) == p.B && t.size(1) == h && t.size(2) == p.T &&
           t.size(3) == kHeadDim;
  };
  return heads(*p.q, p.NH) && heads(*p.k, p.NKV) && heads(*p.v, p.NKV) &&
         (!p.valid || (is(*p.valid, at::kByte, 2, dev) && shape2(*p.valid, p.B, p.T)));
}

// attn_fwd(q, k, v, valid, scale) -> (out, lse)
OP(attn_fwd) {
  HANDLE_TH_ERRORS
  ARGS(5);
  const double scale = PyFloat_AsDouble(a[4]);
  if (PyErr_Occurred()) return nullptr;
  PaddedArgs p;
  if (!padded_args(a, p)) ELSE_PYTHON;
  const at::Device dev = p.q->device();
  Tensor out = empty({p.B * p.T, p.NH * kHeadDim}, at::kHalf, dev);
  Tensor lse = empty({p.B, p.NH, p.T}, at::kFloat, dev);
  void* st = stream_of(out);
  if (!launched("soupk_attention_fwd", [&] {
        return p_soupk_attention_fwd(
            ptr<uint16_t>(p.q), ptr<uint16_t>(p.k), ptr<uint16_t>(p.v), ptr<uint8_t>(p.valid),
            ptr<uint16_t>(out), ptr<float>(lse), static_cast<int32_t>(p.B),
            static_cast<int32_t>(p.T), static_cast<int32_t>(p.NH), static_cast<int32_t>(p.NKV),
            kHeadDim, static_cast<float>(scale), st);
      }))
    return nullptr;
  return pack({out, lse});
  END_HANDLE_TH_ERRORS
}

// attn_bwd(q, k, v, valid, out, lse, dout, scale) -> (dq, dk, dv)
OP(attn_bwd) {
  HANDLE_TH_ERRORS
  ARGS(8);
  const double scale = PyFloat_AsDouble(a[7]);
  if (PyErr_Occurred()) return nullptr;
  PaddedArgs p;
  const Tensor *out = plain(a[4]), *lse = plain(a[5]), *dout = plain(a[6]);
  if (!padded_args(a, p) || !out || !lse || !dout) ELSE_PYTHON;
  const at::Device dev = p.q->device();
  const int64_t BT = p.B * p.T, HD = p.NH * kHeadDim;
  if (!is(*out, at::kHalf, 2, dev) || !shape2(*out, BT, HD) || !is(*dout, at::kHalf, 2, dev) ||
      !shape2(*dout, BT, HD) || !is(*lse, at::kFloat, 3, dev) || lse->size(0) != p.B ||
      lse->size(1) != p.NH || lse->size(2) != p.T)
    ELSE_PYTHON;
  Tensor dq = at::empty_like(*p.q), dk = at::empty_like(*p.k), dv = at::empty_like(*p.v);
  Tensor ws = empty({(p.B * p.NH * p.T + 3) / 4 * 4 + 2 * p.B * p.NH * p.T * kHeadDim}, at::kFloat,
                    dev);
  void* st = stream_of(dq);
  if (!launched("soupk_attention_bwd", [&] {
        return p_soupk_attention_bwd(
            ptr<uint16_t>(p.q), ptr<uint16_t>(p.k), ptr<uint16_t>(p.v), ptr<uint8_t>(p.valid),
            ptr<uint16_t>(out), ptr<uint16_t>(dout), ptr<float>(lse), ptr<float>(ws),
            ptr<uint16_t>(dq), ptr<uint16_t>(dk), ptr<uint16_t>(dv), static_cast<int32_t>(p.B),
            static_cast<int32_t>(p.T), static_cast<int32_t>(p.NH), static_cast<int32_t>(p.NKV),
            kHeadDim, static_cast<float>(scale), st);
      }))
    return nullptr;
  return pack({dq, dk, dv});
  END_HANDLE_TH_ERRORS
}

// swiglu_fwd(gu) -> act
OP(swiglu_fwd) {
  HANDLE_TH_ERRORS
  ARGS(1);
  const Tensor* gu = plain(a[0]);
  if (!gu || gu->dim() != 2 || !is(*gu, at::kHalf, 2, gu->device()) || gu->size(1) % 2 ||
      gu->numel() == 0)
    ELSE_PYTHON;
  const int64_t rows = gu->size(0), inter = gu->size(1) / 2;
  Tensor act = empty({rows, inter}, at::kHalf, gu->device());
  void* st = stream_of(act);
  if (!launched("soupk_swiglu_fwd", [&] {
        return p_soupk_swiglu_fwd(ptr<uint16_t>(gu), ptr<uint16_t>(act), rows, inter, st);
      }))
    return nullptr;
  return THPVariable_Wrap(act);
  END_HANDLE_TH_ERRORS
}

// gemm(a, b, bias, accumulate_out, algo, workspace_bytes) -> out: a [M, K] @ b [K, N] on hipBLASLt
// (blas.matmul's conditions and arguments), into a new [M, N] or added to accumulate_out.
OP(gemm) {
  HANDLE_TH_ERRORS
  ARGS(6);
  const Tensor *x = plain(a[0]), *w = plain(a[1]), *bias, *into;
  if (!x || !w || !optional(a[2], bias) || !optional(a[3], into)) ELSE_PYTHON;
  const int64_t algo = NUM(4), ws_bytes = NUM(5);
  if (PyErr_Occurred()) return nullptr;
  const at::Device dev = x->device();
  auto half2 = [&](const Tensor& t) {
    return t.is_cuda() && t.device() == dev && t.scalar_type() == at::kHalf && t.dim() == 2 &&
           t.layout() == at::kStrided && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
  };
  if (!half2(*x) || !half2(*w)) ELSE_PYTHON;
  const int64_t M = x->size(0), K = x->size(1), N = w->size(1);
  const int64_t xs = x->stride(0), w0 = w->stride(0), w1 = w->stride(1);
  const bool rows = w1 == 1 && (K == 1 || w0 >= N);
  const bool cols = !rows && w0 == 1 && (N == 1 || w1 >= K);
  if (w->size(0) != K || M == 0 || N == 0 || K == 0 || x->stride(1) != 1 || !(rows || cols) ||
      (M > 1 && xs < K) ||
      (bias && (bias->scalar_type() != at::kHalf || !bias->is_contiguous() ||
                bias->numel() != N || into || bias->device() != dev ||
                reinterpret_cast<uintptr_t>(bias->data_ptr()) % 8)) ||
      (into && (!half2(*into) || !shape2(*into, M, N) || into->stride(1) != 1 ||
                (M > 1 && into->stride(0) < N))))
    ELSE_PYTHON;
  const int64_t lda = rows ? std::max(w0, N) : std::max(w1, K), ldb = std::max(xs, K);
  const int64_t ldd = into ? std::max(into->stride(0), N) : N;
  if ((lda | ldb | ldd) % 8) ELSE_PYTHON;
  Tensor out = into ? *into : empty({M, N}, at::kHalf, dev);
  Tensor ws = empty({ws_bytes}, at::kByte, dev);
  void* st = stream_of(*x);
  if (!launched("soupk_gemm_lt", [&] {
        return p_soupk_gemm_lt(rows ? 0 : 1, 0, N, M, K, ptr<uint16_t>(w), lda, 0,
                               ptr<uint16_t>(x), ldb, 0, ptr<uint16_t>(out), ldd, 0, 0, 1,
                               into ? 1 : 0, ptr<uint16_t>(bias), static_cast<int32_t>(algo),
                               ptr(&ws), ws_bytes, st);
      }))
    return nullptr;
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

struct Ref {
  PyObject* o;
  ~Ref() { Py_XDECREF(o); }
};

constexpr int kKeyWords = 6 * 3 + 2 + 3;

// Everything a plan of an NF4 weight is made from and checked on -- for the packed data and each
// state tensor its address, element count, type, device and whether it is contiguous; the same of
// the offset, or its value when it is a number; the shape; both block sizes; whether it is nested
// NF4.  False (no Python error) for an object without that state.
bool weight_key(PyObject* weight, uint64_t* key) {
  static PyObject* const names[] = {
      PyUnicode_InternFromString("quant_state"), PyUnicode_InternFromString("data"),
      PyUnicode_InternFromString("absmax"),      PyUnicode_InternFromString("code"),
      PyUnicode_InternFromString("state2"),      PyUnicode_InternFromString("offset"),
      PyUnicode_InternFromString("shape"),       PyUnicode_InternFromString("blocksize"),
      PyUnicode_InternFromString("quant_type"),  PyUnicode_InternFromString("nested")};
  auto none = [] {
    PyErr_Clear();
    return false;
  };
  auto get = [](PyObject* o, int i) { return Ref{o ? PyObject_GetAttr(o, names[i]) : nullptr}; };
  const Ref state = get(weight, 0);
  if (!state.o) return none();
  const Ref data = get(weight, 1), absmax = get(state.o, 2), code = get(state.o, 3),
            state2 = get(state.o, 4), offset = get(state.o, 5), shape = get(state.o, 6),
            block = get(state.o, 7), type = get(state.o, 8), nested = get(state.o, 9);
  const Ref code2 = get(state2.o, 3), absmax2 = get(state2.o, 2), block2 = get(state2.o, 7);
  if (PyErr_Occurred()) return none();
  auto tensor = [&](PyObject* o) {
    const Tensor& t = THPVariable_Unpack(o);
    const at::Device d = t.device();
    *key++ = reinterpret_cast<uintptr_t>(t.data_ptr());
    *key++ = static_cast<uint64_t>(t.numel());
    *key++ = static_cast<uint64_t>(static_cast<uint8_t>(t.scalar_type())) |
             static_cast<uint64_t>(t.is_contiguous()) << 8 |
             static_cast<uint64_t>(static_cast<uint8_t>(d.type())) << 16 |
             static_cast<uint64_t>(static_cast<uint8_t>(d.index())) << 24;
  };
  for (PyObject* o : {data.o, absmax.o, code.o, code2.o, absmax2.o}) {
    if (!THPVariable_Check(o)) return false;
    tensor(o);
  }
  if (THPVariable_Check(offset.o)) {
    tensor(offset.o);
  } else {
    const double v = PyFloat_AsDouble(offset.o);
    std::memcpy(key, &v, sizeof(v));
    key[1] = key[2] = ~uint64_t{0};        // (no tensor)
    key += 3;
  }
  if (PySequence_Size(shape.o) != 2) return none();
  for (Py_ssize_t d = 0; d < 2; ++d) {
    const Ref n{PySequence_GetItem(shape.o, d)};
    *key++ = n.o ? PyLong_AsUnsignedLongLongMask(n.o) : 0;
  }
  *key++ = PyLong_AsUnsignedLongLongMask(block.o);
  *key++ = PyLong_AsUnsignedLongLongMask(block2.o);
  const int is_nested = PyObject_IsTrue(nested.o);
  *key = (is_nested == 1 ? 1u : 0u) |
         (PyUnicode_Check(type.o) && !PyUnicode_CompareWithASCIIString(type.o, "nf4") ? 2u : 0u);
  return PyErr_Occurred() ? none() : true;
}

// nf4_key(weight) -> bytes (weight_key), None for an object without that state.
OP(nf4_key) {
  HANDLE_TH_ERRORS
  ARGS(1);
  uint64_t key[kKeyWords];
  if (!weight_key(a[0], key)) ELSE_PYTHON;
  return PyBytes_FromStringAndSize(reinterpret_cast<const char*>(key), sizeof(key));
  END_HANDLE_TH_ERRORS
}

// nf4_keys(tuple of weights) -> bytes: their keys one after the other; None when there are none, or
// one has none.
OP(nf4_keys) {
  HANDLE_TH_ERRORS
  ARGS(1);
  if (!PyTuple_Check(a[0])) return PyErr_Format(PyExc_TypeError, "a tuple of weights is expected");
  const Py_ssize_t m = PyTuple_GET_SIZE(a[0]);
  if (m == 0) ELSE_PYTHON;
  const Ref out{PyBytes_FromStringAndSize(nullptr, m * kKeyWords * sizeof(uint64_t))};
  if (!out.o) return nullptr;
  for (Py_ssize_t i = 0; i < m; ++i) {
    uint64_t key[kKeyWords];
    if (!weight_key(PyTuple_GET_ITEM(a[0], i), key)) ELSE_PYTHON;
    std::memcpy(PyBytes_AS_STRING(out.o) + i * sizeof(key), key, sizeof(key));
  }
  return Py_NewRef(out.o);
  END_HANDLE_TH_ERRORS
}

// abi_version() -> the version of soupk.h that this file's function types were compiled from
OP(abi_version) {
  ARGS(0);
  return PyLong_FromLong(SOUPK_ABI_VERSION);
}

// set_status(SoupkError, address of soupk_status_string)
OP(set_status) {
  ARGS(2);
  Py_XDECREF(g_error);
  g_error = Py_NewRef(a[0]);
  p_status_string = reinterpret_cast<const char* (*)(int)>(
      static_cast<uintptr_t>(PyLong_AsUnsignedLongLongMask(a[1])));
  Py_RETURN_NONE;
}

#define M(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(name)), METH_FASTCALL, nullptr}
#define X(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(call_##name)), METH_FASTCALL, nullptr},
PyMethodDef methods[] = {
    SOUPK_ENTRIES(X) M(bind), M(set_status), M(rmsnorm_fwd), M(rmsnorm_bwd), M(rope_tokens),
    M(rope_fwd), M(rope_bwd), M(varlen_fwd), M(varlen_bwd), M(attn_fwd), M(attn_bwd),
    M(swiglu_fwd), M(gemm), M(nf4_key), M(nf4_keys), M(abi_version), {nullptr, nullptr, 0, nullptr}};
#undef X
#undef M

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_soupk_host", nullptr, -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__soupk_host() { return PyModule_Create(&module); }
