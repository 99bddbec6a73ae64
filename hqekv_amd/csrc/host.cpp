// The host side of the per-step and per-layer calls, as a CPython module over torch's C++ tensors.
//
// A decode step of a short or medium cache is three or four launches of a few microseconds each; reading the forty
// fields of a cache tuple, filling the segment tables and building the views of the next tuple from Python took longer
// than the launches ran (a plain call at 1k tokens: 46 us of Python around 7 us of launch calls and 16 us of device
// time).  The functions here do that work on at::Tensor directly.  They take the plain case only -- contiguous device
// tensors of the expected types -- and answer None for anything else, which the Python callers then handle in full.
//
// Kernels are reached through libhqekv's C ABI, bound by path (bind), so that whatever library the package loaded is
// the one used here.
#include <Python.h>
#include <dlfcn.h>
#include <math.h>
#include <stdlib.h>
#include <string.h>

#include <chrono>
#include <initializer_list>
#include <thread>
#include <vector>

#include <ATen/core/Tensor.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <ATen/ops/empty.h>
#include <ATen/core/CachingHostAllocator.h>
#include <hip/hip_runtime_api.h>
#include <c10/core/DeviceGuard.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "hqekv.h"

namespace {

using at::Tensor;

// ------------------------------------------------------------------------------------------------ the C ABI
#define HQ_SYMBOLS(X)             \
  X(hqekv_last_error)             \
  X(hqekv_decode_workspace_bytes) \
  X(hqekv_decode_attn)            \
  X(hqekv_decode_step)            \
  X(hqekv_quant_pack_rows)        \
  X(hqekv_quant_pack_k_tokenmajor)  \
  X(hqekv_prompt_attn)              \
  X(hqekv_prompt_last_rows)         \
  X(hqekv_prompt_last_rows_workspace_bytes) \
  X(hqekv_cache_reconstruct)        \
  X(hqekv_importance_scores)        \
  X(hqekv_weighted_block_scores)    \
  X(hqekv_range_block_scores)       \
  X(hqekv_rank_blocks)              \
  X(hqekv_plan_side)                \
  X(hqekv_fetch_words)              \
  X(hqekv_cache_migrate_both)

struct Api {
#define X(n_) decltype(&::n_) n_ = nullptr;
  HQ_SYMBOLS(X)
#undef X
} api;

PyObject *s_cover, *s_blocks, *s_host_version;   // interned attribute names

// the exceptions of _lib.check
PyObject *raise_rc(int64_t rc, const char *what) {
  const char *msg = api.hqekv_last_error();
  if (rc < 0) return PyErr_Format(PyExc_ValueError, "%s: %s (code %lld)", what, msg, (long long)rc);
  return PyErr_Format(PyExc_RuntimeError, "%s: HIP error %lld: %s", what, (long long)rc, msg);
}

// Other Python threads run while the kernels' library is entered (a launch waits in there when the device's queue is full)
// and while memory is asked for.  `f` touches nothing of Python's, and no field of an object that a second thread may call
// into: those are read before it, into copies that keep tensors alive, and written after it.
struct WithoutGil {
  PyThreadState *state = PyEval_SaveThread();
  ~WithoutGil() { PyEval_RestoreThread(state); }
};
template <typename F>
auto without_gil(F &&f) {
  const WithoutGil others;
  return f();
}

// ------------------------------------------------------------------------------------------------ tensors
bool is_tensor(PyObject *o) { return THPVariable_Check(o); }
const Tensor &ten(PyObject *o) { return THPVariable_Unpack(o); }

bool plain_f16(const Tensor &t, int64_t dim, const at::Device &dev) {
  return t.dim() == dim && t.scalar_type() == at::kHalf && t.device() == dev && t.is_contiguous();
}
bool plain_i32(const Tensor &t, int64_t dim, const at::Device &dev) {
  return t.dim() == dim && t.scalar_type() == at::kInt && t.device() == dev && t.is_contiguous();
}
void *stream_of(const at::Device &dev) {
  return (void *)c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(dev.index()).stream();
}
Tensor new_tensor(at::IntArrayRef shape, at::ScalarType type, const at::Device &dev) {
  return at::empty(shape, at::TensorOptions().dtype(type).device(dev));
}

// Token rows [from, from + n) of a (B, H, capacity, X) buffer: x.slice(2, from, from + n) at a third of its price (a step
// makes up to seven).  The version counter is the buffer's, as a view's is.
Tensor rows_of(const Tensor &x, int64_t from, int64_t n) {
  if (x.requires_grad()) return x.slice(2, from, from + n);
  c10::TensorImpl *base = x.unsafeGetTensorImpl();
  Tensor t = at::detail::make_tensor<c10::TensorImpl>(c10::TensorImpl::VIEW, c10::Storage(x.storage()), x.key_set(), x.dtype());
  c10::TensorImpl *impl = t.unsafeGetTensorImpl();
  const int64_t shape[4] = {x.size(0), x.size(1), n, x.size(3)};
  impl->set_sizes_and_strides(shape, x.strides(), x.storage_offset() + from * x.stride(2));
  if (!x.is_inference()) impl->set_version_counter(base->version_counter());
  return t;
}

// ------------------------------------------------------------------------------------------------ the cache tuple
// Field numbers of the 42-field tuple (hqekv_amd/attention.py): fp16 K 0/1, fp16 V 2/3, then per bit width code, idx,
// scale, zero; 39/40 the fp16 residual.
constexpr int BITS[4] = {8, 4, 2, 1};
constexpr int K_BASE[4] = {4, 12, 20, 28}, V_BASE[4] = {8, 16, 24, 32};
constexpr int RANGES = 38, NEW_K = 39, NEW_V = 40, TUPLE_LEN = 42;

struct Side {
  hqekv_seg seg[HQEKV_MAX_SEGS + 2];
  PyObject *idx[HQEKV_MAX_SEGS];
  int n = 0, n_idx = 0;
  int64_t class_tokens = 0, tokens = 0, H = -1, D = -1;
};

bool same_heads(Side &s, int64_t H, int64_t D) {
  if (s.H < 0) {
    s.H = H;
    s.D = D;
  }
  return s.H == H && s.D == D;
}

bool position_array(PyObject *o, int64_t n, const at::Device &dev, Side &s, hqekv_seg &e) {
  if (!is_tensor(o)) return false;
  const Tensor &t = ten(o);
  if (t.scalar_type() != at::kLong || t.device() != dev || !t.is_contiguous() || t.numel() != n) return false;
  e.idx = (const int64_t *)t.data_ptr();
  s.idx[s.n_idx++] = o;
  return true;
}

// One side of the tuple as a segment table, in launch order; false: something is not plain.  The residual's position
// is filled in by the caller (Tall - its tokens).
bool read_side(PyObject *pkv, bool is_k, bool low_uniform, int64_t B, const at::Device &dev, Side &s) {
  memset(s.seg, 0, sizeof(s.seg));
  PyObject *f16 = PyTuple_GET_ITEM(pkv, is_k ? 0 : 2);
  if (f16 != Py_None) {
    if (!is_tensor(f16)) return false;
    const Tensor &t = ten(f16);
    if (t.dim() != 4 || t.scalar_type() != at::kHalf || t.device() != dev || t.size(0) != B) return false;
    hqekv_seg &e = s.seg[s.n++];
    e.bits = 16;
    const int64_t n = t.size(is_k ? 3 : 2), D = t.size(is_k ? 2 : 3), H = t.size(1);
    if (!t.is_contiguous()) {
      // fp16 keys may be the transposed view of token-major memory
      if (!is_k || t.stride(2) != 1 || t.stride(3) != D || t.stride(1) != n * D || (B > 1 && t.stride(0) != H * n * D)) return false;
      e.layout = HQEKV_LAYOUT_TOKEN_MAJOR;
    }
    e.n_tokens = n;
    e.data = t.data_ptr();
    if (!same_heads(s, H, D) || !position_array(PyTuple_GET_ITEM(pkv, is_k ? 1 : 3), n, dev, s, e)) return false;
    s.class_tokens += n;
  }
  for (int c = 0; c < 4; ++c) {
    const int base = is_k ? K_BASE[c] : V_BASE[c], bits = BITS[c];
    PyObject *code = PyTuple_GET_ITEM(pkv, base);
    if (code == Py_None) continue;
    PyObject *sc = PyTuple_GET_ITEM(pkv, base + 2), *zr = PyTuple_GET_ITEM(pkv, base + 3);
    if (!is_tensor(code) || !is_tensor(sc) || !is_tensor(zr)) return false;
    const Tensor &tc = ten(code), &ts = ten(sc), &tz = ten(zr);
    if (!plain_i32(tc, 4, dev) || !plain_f16(ts, 4, dev) || !plain_f16(tz, 4, dev) || tc.size(0) != B) return false;
    hqekv_seg &e = s.seg[s.n++];
    const int64_t per = 32 / bits;
    const int64_t n = is_k ? tc.size(3) * per : tc.size(2), D = is_k ? tc.size(2) : tc.size(3) * per;
    if (ts.numel() * 32 != tc.numel() * per || tz.numel() != ts.numel()) return false;
    e.bits = bits;
    e.layout = bits == 1 && !low_uniform ? HQEKV_LAYOUT_NORMAL1 : 0;
    e.n_tokens = n;
    e.data = tc.data_ptr();
    e.scale = ts.data_ptr();
    e.zero = tz.data_ptr();
    if (!same_heads(s, tc.size(1), D) || !position_array(PyTuple_GET_ITEM(pkv, base + 1), n, dev, s, e)) return false;
    s.class_tokens += n;
  }
  s.tokens = s.class_tokens;
  PyObject *res = PyTuple_GET_ITEM(pkv, is_k ? NEW_K : NEW_V);
  if (res != Py_None) {
    if (!is_tensor(res)) return false;
    const Tensor &t = ten(res);
    if (t.dim() != 4 || t.scalar_type() != at::kHalf || t.device() != dev || t.size(0) != B) return false;
    const int64_t H = t.size(1), n = t.size(2), D = t.size(3);
    if (n > 0) {
      hqekv_seg &e = s.seg[s.n++];
      e.bits = 16;
      e.layout = is_k ? HQEKV_LAYOUT_TOKEN_MAJOR : 0;
      e.n_tokens = n;
      e.data = t.data_ptr();
      if (!t.is_contiguous()) {   // the head of a longer buffer
        const int64_t sb = t.stride(0), sh = t.stride(1);
        if (t.stride(3) != 1 || t.stride(2) != D || sh % D || sh < n * D || (B > 1 && sb != H * sh)) return false;
        e.slab_tokens = sh / D;
      }
      if (!same_heads(s, H, D)) return false;
      s.tokens += n;
    }
  }
  return s.n <= HQEKV_MAX_SEGS;
}

// attention.idx_cover_once: the remembered verdict when it still holds for these very arrays, else the function itself
// (which remembers).  -> 3 (covered, in whole runs of 32 positions), 1 (covered), 0, or -1 with an exception set.
int cover_once(PyObject *const *idx, int n_idx, int64_t n, PyObject *cover_fn, bool again = true) {
  if (n_idx == 0) return n == 0 ? 1 : 0;
  PyObject *hit = PyObject_GetAttr(idx[0], s_cover);
  if (!hit) {
    if (!PyErr_ExceptionMatches(PyExc_AttributeError)) return -1;
    PyErr_Clear();
  } else {
    int verdict = -1;
    if (PyTuple_Check(hit) && PyTuple_GET_SIZE(hit) == 4) {
      PyObject *key = PyTuple_GET_ITEM(hit, 0), *refs = PyTuple_GET_ITEM(hit, 2);
      bool ok = PyTuple_Check(key) && PyTuple_GET_SIZE(key) == n_idx + 1 && PyList_Check(refs) && PyList_GET_SIZE(refs) == n_idx &&
                PyLong_AsLongLong(PyTuple_GET_ITEM(key, n_idx)) == n;
      for (int i = 0; ok && i < n_idx; ++i) {
        const Tensor &t = ten(idx[i]);
        PyObject *k = PyTuple_GET_ITEM(key, i);
        ok = PyTuple_Check(k) && PyTuple_GET_SIZE(k) == 3 && !t.is_inference() &&
             PyLong_AsUnsignedLongLongMask(PyTuple_GET_ITEM(k, 0)) == (unsigned long long)(uintptr_t)t.data_ptr() &&
             PyLong_AsLongLong(PyTuple_GET_ITEM(k, 1)) == t.numel() && PyLong_AsLongLong(PyTuple_GET_ITEM(k, 2)) == (long long)t._version() &&
             PyWeakref_Check(PyList_GET_ITEM(refs, i)) && PyWeakref_GET_OBJECT(PyList_GET_ITEM(refs, i)) == idx[i];
      }
      if (ok) verdict = PyTuple_GET_ITEM(hit, 1) != Py_True ? 0 : PyTuple_GET_ITEM(hit, 3) == Py_True ? 3 : 1;
    }
    Py_DECREF(hit);
    if (PyErr_Occurred()) return -1;
    if (verdict >= 0) return verdict;
  }
  PyObject *list = PyList_New(n_idx);
  if (!list) return -1;
  for (int i = 0; i < n_idx; ++i) {
    Py_INCREF(idx[i]);
    PyList_SET_ITEM(list, i, idx[i]);
  }
  PyObject *r = PyObject_CallFunction(cover_fn, "NL", list, (long long)n);
  if (!r) return -1;
  const int v = PyObject_IsTrue(r);
  Py_DECREF(r);
  return v > 0 && again ? cover_once(idx, n_idx, n, cover_fn, false) : v;   // (once more for what it remembered)
}

int default_flags() {
  const char *v = getenv("HQEKV_UNFUSED");
  return v && !strcmp(v, "1") ? 0 : HQEKV_FUSE_SOFTMAX;
}

// ------------------------------------------------------------------------------------------------ decode
// decode(q, pkv, low_uniform, cover_fn) -> (attn_weights, attn_output), or None where the call is not plain
PyObject *decode(PyObject *, PyObject *const *a, Py_ssize_t na) {
  HANDLE_TH_ERRORS
  if (na != 4) return PyErr_Format(PyExc_TypeError, "decode takes 4 arguments");
  PyObject *pkv = a[1];
  const int flags = default_flags();
  if (!is_tensor(a[0]) || !PyTuple_Check(pkv) || PyTuple_GET_SIZE(pkv) != TUPLE_LEN || !flags) Py_RETURN_NONE;
  const Tensor &q = ten(a[0]);
  if (!q.is_cuda() || q.dim() != 4 || q.scalar_type() != at::kHalf || q.size(2) != 1 || !q.is_contiguous()) Py_RETURN_NONE;
  const at::Device dev = q.device();
  const int64_t B = q.size(0), Hq = q.size(1), D = q.size(3);
  Side k, v;
  const bool low_uniform = a[2] == Py_True;
  if (!read_side(pkv, true, low_uniform, B, dev, k) || !read_side(pkv, false, low_uniform, B, dev, v)) Py_RETURN_NONE;
  const int64_t Tall = v.tokens;
  if (Tall == 0 || k.tokens != Tall || k.class_tokens != v.class_tokens || k.H != v.H || k.D != D || v.D != D) Py_RETURN_NONE;
  for (Side *s : {&k, &v}) {
    const int c = cover_once(s->idx, s->n_idx, v.class_tokens, a[3]);
    if (c < 0) return nullptr;
    if (!c) Py_RETURN_NONE;
    for (int i = 0; c == 3 && i < s->n; ++i)
      if (s->seg[i].idx) s->seg[i].layout |= HQEKV_LAYOUT_RUNS;
  }
  for (Side *s : {&k, &v})
    if (s->tokens > s->class_tokens) s->seg[s->n - 1].pos_base = s->class_tokens;
  const c10::OptionalDeviceGuard guard(dev);
  const int64_t need = api.hqekv_decode_workspace_bytes(k.seg, k.n, v.seg, v.n, B, Hq, k.H, D);
  if (need < 0) return PyErr_Format(PyExc_ValueError, "invalid segment table");
  Tensor weights, out;
  const int rc = without_gil([&] {
    weights = new_tensor({B, Hq, 1, Tall}, at::kHalf, dev);
    out = new_tensor({B, Hq, 1, D}, at::kHalf, dev);
    const Tensor ws = new_tensor({std::max<int64_t>(need, 256)}, at::kByte, dev);
    return api.hqekv_decode_attn(k.seg, k.n, v.seg, v.n, q.data_ptr(), nullptr, 0, weights.data_ptr(), out.data_ptr(), B, Hq, k.H, D, Tall,
                                 ws.data_ptr(), ws.numel(), flags, stream_of(dev));
  });
  if (rc) return raise_rc(rc, "decode_attention");
  return Py_BuildValue("NN", THPVariable_Wrap(weights), THPVariable_Wrap(out));
  END_HANDLE_TH_ERRORS
}

// ------------------------------------------------------------------------------------------------ a layer's steps
// The class entries of a layer's segment tables between two compressions, with room for the residual and the step's own
// token, and the workspace of its steps.
struct StepTables {
  PyObject_HEAD
  hqekv_seg k[HQEKV_MAX_SEGS], v[HQEKV_MAX_SEGS];
  int n_k, n_v;
  Tensor ws;
};

PyObject *tables_new(PyTypeObject *type, PyObject *args, PyObject *) {
  unsigned long long ka, va;
  int nk, nv;
  if (!PyArg_ParseTuple(args, "KiKi", &ka, &nk, &va, &nv)) return nullptr;
  if (nk < 0 || nv < 0 || nk > HQEKV_MAX_SEGS - 2 || nv > HQEKV_MAX_SEGS - 2) return PyErr_Format(PyExc_ValueError, "too many segments");
  StepTables *t = (StepTables *)type->tp_alloc(type, 0);
  if (!t) return nullptr;
  memset(t->k, 0, sizeof(t->k));
  memset(t->v, 0, sizeof(t->v));
  memcpy(t->k, (const void *)(uintptr_t)ka, nk * sizeof(hqekv_seg));
  memcpy(t->v, (const void *)(uintptr_t)va, nv * sizeof(hqekv_seg));
  t->n_k = nk;
  t->n_v = nv;
  new (&t->ws) Tensor();
  return (PyObject *)t;
}
// step_tables(q, pkv, low_uniform, cover_fn) -> StepTables over the tuple's classes -- they have to cover every position
// once --, or None where the tuple is not plain.  The caller keeps the class tensors.  (Built from Python's segment lists
// they cost the first step after a compression 47 us: a prompt of 1024 tokens and 24 steps 434 -> 387 us; behind a longer
// prompt's attention it is hidden, 4099 tokens 488 -> 486.)
PyTypeObject *tables_type_ptr();
PyObject *step_tables(PyObject *, PyObject *const *a, Py_ssize_t na) {
  HANDLE_TH_ERRORS
  if (na != 4) return PyErr_Format(PyExc_TypeError, "step_tables takes 4 arguments");
  PyObject *pkv = a[1];
  if (!is_tensor(a[0]) || !PyTuple_Check(pkv) || PyTuple_GET_SIZE(pkv) != TUPLE_LEN) Py_RETURN_NONE;
  const Tensor &q = ten(a[0]);
  if (!q.is_cuda() || q.dim() != 4) Py_RETURN_NONE;
  const at::Device dev = q.device();
  const int64_t B = q.size(0);
  const bool low_uniform = a[2] == Py_True;
  Side k, v;
  if (!read_side(pkv, true, low_uniform, B, dev, k) || !read_side(pkv, false, low_uniform, B, dev, v)) Py_RETURN_NONE;
  if (!v.class_tokens || k.class_tokens != v.class_tokens || k.H != v.H || k.D != v.D || k.n_idx > HQEKV_MAX_SEGS - 2 || v.n_idx > HQEKV_MAX_SEGS - 2)
    Py_RETURN_NONE;
  for (Side *s : {&k, &v}) {
    const int c = cover_once(s->idx, s->n_idx, v.class_tokens, a[3]);
    if (c < 0) return nullptr;
    if (!c) Py_RETURN_NONE;
    for (int i = 0; c == 3 && i < s->n_idx; ++i) s->seg[i].layout |= HQEKV_LAYOUT_RUNS;
  }
  StepTables *t = (StepTables *)tables_type_ptr()->tp_alloc(tables_type_ptr(), 0);
  if (!t) return nullptr;
  memset(t->k, 0, sizeof(t->k));
  memset(t->v, 0, sizeof(t->v));
  memcpy(t->k, k.seg, k.n_idx * sizeof(hqekv_seg));   // (the classes come first, one position array each)
  memcpy(t->v, v.seg, v.n_idx * sizeof(hqekv_seg));
  t->n_k = k.n_idx;
  t->n_v = v.n_idx;
  new (&t->ws) Tensor();
  return (PyObject *)t;
  END_HANDLE_TH_ERRORS
}
void tables_free(PyObject *o) {
  ((StepTables *)o)->ws.~Tensor();
  Py_TYPE(o)->tp_free(o);
}

void f16_rows(hqekv_seg &e, int layout, int64_t n, int64_t pos, const void *data, int64_t slab) {
  e = hqekv_seg{};
  e.bits = 16;
  e.layout = layout;
  e.n_tokens = n;
  e.pos_base = pos;
  e.data = data;
  e.slab_tokens = slab;
}

// The attention call of a step, with the workspace kept from step to step (twice what is needed when it is made: room
// for the residual to grow without asking again).  The tables are the caller's own copies.
int run_step(const hqekv_seg *k, int n_k, const hqekv_seg *v, int n_v, const Tensor &q, const Tensor &weights, const Tensor &out,
             int64_t Hkv, int64_t Tall, Tensor &kept, const at::Device &dev, const hqekv_step_extra *x) {
  const int64_t B = q.size(0), Hq = q.size(1), D = q.size(3);
  const int flags = default_flags();
  Tensor ws = kept;
  const int rc = without_gil([&] {
    auto call = [&]() -> int {
      return api.hqekv_decode_step(k, n_k, v, n_v, q.data_ptr(), nullptr, 0, weights.data_ptr(), out.data_ptr(), B, Hq, Hkv, D, Tall,
                                   ws.data_ptr(), ws.numel(), flags, stream_of(dev), x);
    };
    if (ws.defined() && ws.device() == dev) {
      const int rc = call();
      if (rc != HQEKV_E_WORKSPACE) return rc;   // else the cache has outgrown the workspace of earlier steps
    }
    const int64_t need = api.hqekv_decode_workspace_bytes(k, n_k, v, n_v, B, Hq, Hkv, D);
    if (need < 0) return (int)HQEKV_E_ARG;
    ws = new_tensor({std::max<int64_t>(2 * need, 256)}, at::kByte, dev);
    return call();
  });
  kept = ws;
  return rc;
}

bool step_inputs(const Tensor &q, const Tensor &k, const Tensor &v, int64_t D) {
  if (!q.is_cuda() || !plain_f16(q, 4, q.device()) || q.size(2) != 1 || q.size(3) != D) return false;
  for (const Tensor *t : {&k, &v})
    if (!plain_f16(*t, 4, q.device()) || t->size(0) != q.size(0) || t->size(2) != 1 || t->size(3) != D) return false;
  return k.size(1) == v.size(1);
}

// StepTables.step(q, k, v, pkv, kbuf, vbuf, n, Tall, ring_store, ring_row, kv_seq_len): one decode step whose classes
// cover every position once.  The residual is the first n token rows of the capacity buffers, k and v follow it as a
// segment of their own and are copied to row n by the call's last launch; row `ring_row` of ring_store (None: no ring)
// receives the ring row.  -> (attn_weights, attn_output, the next tuple), or None where the inputs are not plain.
PyObject *tables_step(PyObject *self, PyObject *const *a, Py_ssize_t na) {
  HANDLE_TH_ERRORS
  if (na != 11) return PyErr_Format(PyExc_TypeError, "step takes 11 arguments");
  StepTables *s = (StepTables *)self;
  for (int i : {0, 1, 2, 4, 5})
    if (!is_tensor(a[i])) Py_RETURN_NONE;
  const Tensor &q = ten(a[0]), &k = ten(a[1]), &v = ten(a[2]), &kb = ten(a[4]), &vb = ten(a[5]);
  PyObject *pkv = a[3];
  const int64_t n = PyLong_AsLongLong(a[6]), Tall = PyLong_AsLongLong(a[7]), row = PyLong_AsLongLong(a[9]);
  if (PyErr_Occurred()) return nullptr;
  const int64_t D = kb.dim() == 4 ? kb.size(3) : 0;
  if (!step_inputs(q, k, v, D) || !PyTuple_Check(pkv) || PyTuple_GET_SIZE(pkv) != TUPLE_LEN) Py_RETURN_NONE;
  const at::Device dev = q.device();
  for (const Tensor *b : {&kb, &vb})
    if (!plain_f16(*b, 4, dev) || b->size(0) != q.size(0) || b->size(1) != k.size(1) || b->size(3) != D || n < 0 || n >= b->size(2)) Py_RETURN_NONE;
  hqekv_step_extra x{};
  if (a[8] != Py_None) {
    if (!is_tensor(a[8])) Py_RETURN_NONE;
    const Tensor &ring = ten(a[8]);
    if (!plain_f16(ring, 2, dev) || row < 0 || row >= ring.size(0) || ring.size(1) < Tall) Py_RETURN_NONE;
    x.ring_line = (char *)ring.data_ptr() + 2 * row * ring.size(1);
  }
  const int64_t cap_k = kb.size(2), cap_v = vb.size(2);
  int n_k = s->n_k, n_v = s->n_v;
  hqekv_seg ks[HQEKV_MAX_SEGS], vs[HQEKV_MAX_SEGS];
  memcpy(ks, s->k, n_k * sizeof(hqekv_seg));
  memcpy(vs, s->v, n_v * sizeof(hqekv_seg));
  if (n) {
    f16_rows(ks[n_k++], HQEKV_LAYOUT_TOKEN_MAJOR, n, Tall - 1 - n, kb.data_ptr(), cap_k);
    f16_rows(vs[n_v++], 0, n, Tall - 1 - n, vb.data_ptr(), cap_v);
  }
  f16_rows(ks[n_k++], HQEKV_LAYOUT_TOKEN_MAJOR, 1, Tall - 1, k.data_ptr(), 0);
  f16_rows(vs[n_v++], 0, 1, Tall - 1, v.data_ptr(), 0);
  const c10::OptionalDeviceGuard guard(dev);
  Tensor weights = new_tensor({q.size(0), q.size(1), 1, Tall}, at::kHalf, dev), out = new_tensor({q.size(0), q.size(1), 1, D}, at::kHalf, dev);
  // (how torch's reduction deals the head rows to threads: attention.ring_order)
  x.ring_order = Tall % 4 == 0 && Tall >= 256 && (uintptr_t)weights.data_ptr() % 8 == 0 ? 2 : 1;
  x.append_rows = 1;
  x.new_k = k.data_ptr();
  x.new_v = v.data_ptr();
  x.k_dst = (char *)kb.data_ptr() + 2 * D * n;
  x.v_dst = (char *)vb.data_ptr() + 2 * D * n;
  x.k_dst_slab_tokens = cap_k;
  x.v_dst_slab_tokens = cap_v;
  const int rc = run_step(ks, n_k, vs, n_v, q, weights, out, k.size(1), Tall, s->ws, dev, &x);
  if (rc) return raise_rc(rc, "decode_step");
  PyObject *next = PyTuple_New(TUPLE_LEN);
  if (!next) return nullptr;
  for (int i = 0; i < NEW_K; ++i) {
    PyObject *o = PyTuple_GET_ITEM(pkv, i);
    Py_INCREF(o);
    PyTuple_SET_ITEM(next, i, o);
  }
  PyTuple_SET_ITEM(next, NEW_K, THPVariable_Wrap(rows_of(kb, 0, n + 1)));
  PyTuple_SET_ITEM(next, NEW_V, THPVariable_Wrap(rows_of(vb, 0, n + 1)));
  Py_INCREF(a[10]);
  PyTuple_SET_ITEM(next, TUPLE_LEN - 1, a[10]);
  return Py_BuildValue("NNN", THPVariable_Wrap(weights), THPVariable_Wrap(out), next);
  END_HANDLE_TH_ERRORS
}

PyMethodDef tables_methods[] = {
    {"step", (PyCFunction)(void (*)(void))tables_step, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyTypeObject tables_type = {PyVarObject_HEAD_INIT(nullptr, 0)};
PyTypeObject *tables_type_ptr() { return &tables_type; }

// What KiviAttentionLayer keeps between two decode steps: the K class, the fp16 K tail in a buffer of residual_length
// rows, the V tail as a window [v0, v0 + nv) of a longer buffer, the V class in capacity buffers, and the tuple (views of
// all this) it handed out last.
struct KiviState {
  PyObject_HEAD
  Tensor kq, ks, kz, kt, vt, vcode, vscale, vzero, ws;
  int64_t nk, v0, nv, n_vq;
  PyObject *returned;   // the tuple handed out last
};

PyObject *kivi_new(PyTypeObject *type, PyObject *, PyObject *) {
  KiviState *s = (KiviState *)type->tp_alloc(type, 0);
  if (!s) return nullptr;
  for (Tensor *t : {&s->kq, &s->ks, &s->kz, &s->kt, &s->vt, &s->vcode, &s->vscale, &s->vzero, &s->ws}) new (t) Tensor();
  s->nk = s->v0 = s->nv = s->n_vq = 0;
  Py_INCREF(Py_None);
  s->returned = Py_None;
  return (PyObject *)s;
}
void kivi_free(PyObject *o) {
  KiviState *s = (KiviState *)o;
  for (Tensor *t : {&s->kq, &s->ks, &s->kz, &s->kt, &s->vt, &s->vcode, &s->vscale, &s->vzero, &s->ws}) t->~Tensor();
  Py_CLEAR(s->returned);
  Py_TYPE(o)->tp_free(o);
}

template <Tensor KiviState::*F>
PyObject *kivi_get(PyObject *o, void *) {
  const Tensor &t = ((KiviState *)o)->*F;
  if (!t.defined()) Py_RETURN_NONE;
  return THPVariable_Wrap(t);
}
template <Tensor KiviState::*F>
int kivi_set(PyObject *o, PyObject *v, void *) {
  if (!v || (v != Py_None && !is_tensor(v))) {
    PyErr_SetString(PyExc_TypeError, "a tensor or None");
    return -1;
  }
  ((KiviState *)o)->*F = v == Py_None ? Tensor() : ten(v);
  return 0;
}
template <int64_t KiviState::*F>
PyObject *kivi_get_int(PyObject *o, void *) {
  return PyLong_FromLongLong(((KiviState *)o)->*F);
}
template <int64_t KiviState::*F>
int kivi_set_int(PyObject *o, PyObject *v, void *) {
  const long long n = v ? PyLong_AsLongLong(v) : -1;
  if (n < 0) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "a count");
    return -1;
  }
  ((KiviState *)o)->*F = n;
  return 0;
}
PyObject *kivi_get_returned(PyObject *o, void *) {
  PyObject *r = ((KiviState *)o)->returned;
  Py_INCREF(r);
  return r;
}
PyGetSetDef kivi_fields[] = {
#define F(n_) {#n_, kivi_get<&KiviState::n_>, kivi_set<&KiviState::n_>, nullptr, nullptr}
    F(kq), F(ks), F(kz), F(kt), F(vt), F(vcode), F(vscale), F(vzero),
#undef F
#define F(n_) {#n_, kivi_get_int<&KiviState::n_>, kivi_set_int<&KiviState::n_>, nullptr, nullptr}
    F(nk), F(v0), F(nv), F(n_vq),
#undef F
    {"returned", kivi_get_returned, nullptr, nullptr, nullptr},
    {nullptr, nullptr, nullptr, nullptr, nullptr},
};

// KiviState.step(q, k, v, T, k_bits, v_bits): the attention over (K class, K tail, this step's key) and (V class, V tail,
// this step's value); the call's last launch appends the two rows behind their tails and -- when the tail is full --
// quantises the oldest value row into the class buffers, which must have room for it.  Leaves a full K tail
// (nk == its capacity) and a V window at the end of its buffer to the caller.  -> (attn_weights, attn_output) or None.
PyObject *kivi_step(PyObject *self, PyObject *const *a, Py_ssize_t na) {
  HANDLE_TH_ERRORS
  if (na != 6) return PyErr_Format(PyExc_TypeError, "step takes 6 arguments");
  KiviState *s = (KiviState *)self;
  for (int i : {0, 1, 2})
    if (!is_tensor(a[i])) Py_RETURN_NONE;
  const Tensor &q = ten(a[0]), &k = ten(a[1]), &v = ten(a[2]);
  const int64_t T = PyLong_AsLongLong(a[3]);
  const int k_bits = (int)PyLong_AsLong(a[4]), v_bits = (int)PyLong_AsLong(a[5]);
  if (PyErr_Occurred()) return nullptr;
  if (!s->kt.defined() || !s->vt.defined() || !s->vcode.defined()) return PyErr_Format(PyExc_ValueError, "no buffers");
  const int64_t D = s->kt.size(3), Hkv = s->kt.size(1), R = s->kt.size(2), cap_v = s->vt.size(2), row = 2 * D;
  if (!step_inputs(q, k, v, D) || k.size(1) != Hkv) Py_RETURN_NONE;
  const bool leaves = s->nv + 1 > R;   // a value row leaves the tail after this step
  const int64_t n_kq = s->kq.defined() ? s->kq.size(3) * (32 / k_bits) : 0;
  if (s->nk >= R || s->v0 + s->nv >= cap_v || s->n_vq + leaves > s->vcode.size(2) || n_kq + s->nk + 1 != T || s->n_vq + s->nv + 1 != T ||
      s->kt.size(0) != q.size(0))
    return PyErr_Format(PyExc_ValueError, "KiviAttentionLayer: the buffers do not hold the sequence before this step");
  const at::Device dev = q.device();
  const Tensor held[] = {s->kq, s->ks, s->kz, s->kt, s->vt, s->vcode, s->vscale, s->vzero};
  hqekv_seg ks[3] = {}, vs[3] = {};
  int n_k = 0, n_v = 0;
  if (n_kq) {
    hqekv_seg &e = ks[n_k++];
    e.bits = k_bits;
    e.n_tokens = n_kq;
    e.data = s->kq.data_ptr();
    e.scale = s->ks.data_ptr();
    e.zero = s->kz.data_ptr();
  }
  if (s->nk) f16_rows(ks[n_k++], HQEKV_LAYOUT_TOKEN_MAJOR, s->nk, n_kq, s->kt.data_ptr(), R);
  f16_rows(ks[n_k++], HQEKV_LAYOUT_TOKEN_MAJOR, 1, T - 1, k.data_ptr(), 0);
  if (s->n_vq) {
    hqekv_seg &e = vs[n_v++];
    e.bits = v_bits;
    e.n_tokens = s->n_vq;
    e.data = s->vcode.data_ptr();
    e.scale = s->vscale.data_ptr();
    e.zero = s->vzero.data_ptr();
    e.slab_tokens = s->vcode.size(2);
  }
  char *vt = (char *)s->vt.data_ptr();
  if (s->nv) f16_rows(vs[n_v++], 0, s->nv, s->n_vq, vt + s->v0 * row, cap_v);
  f16_rows(vs[n_v++], 0, 1, T - 1, v.data_ptr(), 0);
  hqekv_step_extra x{};
  x.append_rows = 1;
  x.new_k = k.data_ptr();
  x.new_v = v.data_ptr();
  x.k_dst = (char *)s->kt.data_ptr() + s->nk * row;
  x.v_dst = vt + (s->v0 + s->nv) * row;
  x.k_dst_slab_tokens = R;
  x.v_dst_slab_tokens = cap_v;
  if (leaves) {   // (R > nk >= 0, so the tail has a row: not the one this step appends)
    const int64_t n = s->n_vq, groups = s->vscale.size(3);
    x.leave_bits = v_bits;
    x.leave_src = vt + s->v0 * row;
    x.leave_slab_tokens = cap_v;
    x.leave_code = (char *)s->vcode.data_ptr() + n * s->vcode.size(3) * 4;
    x.leave_scale = (char *)s->vscale.data_ptr() + n * groups * 2;
    x.leave_zero = (char *)s->vzero.data_ptr() + n * groups * 2;
    x.leave_dst_slab_tokens = s->vcode.size(2);
  }
  const c10::OptionalDeviceGuard guard(dev);
  Tensor weights = new_tensor({q.size(0), q.size(1), 1, T}, at::kHalf, dev), out = new_tensor({q.size(0), q.size(1), 1, D}, at::kHalf, dev);
  int rc = run_step(ks, n_k, vs, n_v, q, weights, out, Hkv, T, s->ws, dev, &x);
  if (rc) return raise_rc(rc, "KiviAttentionLayer");
  s->nk += 1;
  s->nv += 1;
  if (leaves) {
    s->n_vq += 1;
    s->v0 += 1;
    s->nv -= 1;
  }
  return Py_BuildValue("NN", THPVariable_Wrap(weights), THPVariable_Wrap(out));
  END_HANDLE_TH_ERRORS
}

// KiviState.fields(T): the 9-field tuple of views over the buffers, remembered as the one handed out last
PyObject *kivi_tuple(PyObject *self, PyObject *T) {
  HANDLE_TH_ERRORS
  KiviState *s = (KiviState *)self;
  auto put = [](PyObject *t, int i, const Tensor &x) {
    if (x.defined()) {
      PyTuple_SET_ITEM(t, i, THPVariable_Wrap(x));
    } else {
      Py_INCREF(Py_None);
      PyTuple_SET_ITEM(t, i, Py_None);
    }
  };
  auto head = [](const Tensor &x, int64_t n) { return n ? rows_of(x, 0, n) : Tensor(); };
  PyObject *t = PyTuple_New(9);
  if (!t) return nullptr;
  put(t, 0, s->kq);
  put(t, 1, head(s->kt, s->nk));
  put(t, 2, s->ks);
  put(t, 3, s->kz);
  put(t, 4, head(s->vcode, s->n_vq));
  put(t, 5, rows_of(s->vt, s->v0, s->nv));
  put(t, 6, head(s->vscale, s->n_vq));
  put(t, 7, head(s->vzero, s->n_vq));
  Py_INCREF(T);
  PyTuple_SET_ITEM(t, 8, T);
  Py_INCREF(t);
  Py_SETREF(s->returned, t);
  return t;
  END_HANDLE_TH_ERRORS
}

PyMethodDef kivi_methods[] = {
    {"step", (PyCFunction)(void (*)(void))kivi_step, METH_FASTCALL, nullptr},
    {"fields", kivi_tuple, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyTypeObject kivi_type = {PyVarObject_HEAD_INIT(nullptr, 0)};

// ------------------------------------------------------------------------------------------------ quantise and pack
// quantize_into(data, bits, code, scale, mn) -> True, or None where a tensor is not plain (pack_unpack.quantize_pack_into)
PyObject *quantize_into(PyObject *, PyObject *const *a, Py_ssize_t na) {
  HANDLE_TH_ERRORS
  if (na != 5) return PyErr_Format(PyExc_TypeError, "quantize_into takes 5 arguments");
  for (int i : {0, 2, 3, 4})
    if (!is_tensor(a[i])) Py_RETURN_NONE;
  const Tensor &x = ten(a[0]), &code = ten(a[2]), &sc = ten(a[3]), &mn = ten(a[4]);
  const int bits = (int)PyLong_AsLong(a[1]);
  if (PyErr_Occurred()) return nullptr;
  if (bits != 1 && bits != 2 && bits != 4 && bits != 8) Py_RETURN_NONE;
  if (!x.is_cuda() || x.dim() != 4 || x.scalar_type() != at::kHalf || code.scalar_type() != at::kInt || sc.scalar_type() != at::kHalf ||
      mn.scalar_type() != at::kHalf || !x.numel())
    Py_RETURN_NONE;
  const at::Device dev = x.device();
  const int64_t B = x.size(0), H = x.size(1), R = x.size(2), L = x.size(3);
  if (L % 32) Py_RETURN_NONE;
  for (const Tensor *t : {&code, &sc, &mn}) {
    if (t->dim() != 4 || t->device() != dev || t->size(0) != B || t->size(1) != H || t->size(2) != R || t->stride(3) != 1 ||
        t->size(3) != (t == &code ? L * bits / 32 : L / 32) || t->stride(0) != H * t->stride(1))
      Py_RETURN_NONE;
  }
  if (sc.stride(1) != mn.stride(1) || sc.stride(2) != mn.stride(2) || sc.stride(0) != mn.stride(0)) Py_RETURN_NONE;
  // read in place: equally spaced (b, h) slabs of dense rows -- or, seen transposed, of dense token rows: the head of a
  // longer tensor is not copied (the stride of a dimension of one element says nothing: it is not looked at)
  const int64_t slab = H > 1 ? x.stride(1) : B > 1 ? x.stride(0) : R * L;
  if ((B > 1 && H > 1 && x.stride(0) != H * slab) || slab < R * L) Py_RETURN_NONE;
  const bool token_major = x.stride(2) == 1 && x.stride(3) == R && R % 2 == 0 && R > 1 && slab % 2 == 0 && (uintptr_t)x.data_ptr() % 4 == 0;
  const bool rows = x.stride(3) == 1 && (R == 1 || x.stride(2) == L) && slab % 8 == 0 && (uintptr_t)x.data_ptr() % 16 == 0;
  if (!token_major && !rows) Py_RETURN_NONE;
  const c10::OptionalDeviceGuard guard(dev);
  const int rc = without_gil([&] {
    return token_major ? api.hqekv_quant_pack_k_tokenmajor(x.data_ptr(), slab, R, code.data_ptr(), code.stride(1), code.stride(2), sc.data_ptr(),
                                                           mn.data_ptr(), sc.stride(1), sc.stride(2), B * H, L, R, bits, stream_of(dev))
                       : api.hqekv_quant_pack_rows(x.data_ptr(), slab, L, code.data_ptr(), code.stride(1), code.stride(2), sc.data_ptr(),
                                                   mn.data_ptr(), sc.stride(1), sc.stride(2), B * H, R, L, bits, stream_of(dev));
  });
  if (rc) return raise_rc(rc, "uniform_group_quantize_pack_last_dim");
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// ------------------------------------------------------------------------------------------------ prompt
bool prompt_rows(const Tensor &t, const at::Device &dev, int64_t (&st)[3]) {
  if (t.dim() != 4 || t.scalar_type() != at::kHalf || t.device() != dev || t.size(3) != 128 || t.stride(3) != 1 || (uintptr_t)t.data_ptr() % 16) return false;
  for (int i = 0; i < 3; ++i) {
    st[i] = t.stride(i);
    if (st[i] % 8) return false;
  }
  return true;
}

// prompt_attention(q, k, v, scaling, causal) -> (B, Hq, T, 128), or None where rows would have to be copied first
PyObject *prompt_attention(PyObject *, PyObject *const *a, Py_ssize_t na) {
  HANDLE_TH_ERRORS
  if (na != 5) return PyErr_Format(PyExc_TypeError, "prompt_attention takes 5 arguments");
  for (int i : {0, 1, 2})
    if (!is_tensor(a[i])) Py_RETURN_NONE;
  const Tensor &q = ten(a[0]), &k = ten(a[1]), &v = ten(a[2]);
  const double scaling = PyFloat_AsDouble(a[3]);
  if (PyErr_Occurred()) return nullptr;
  if (!q.is_cuda()) Py_RETURN_NONE;
  const at::Device dev = q.device();
  int64_t sq[3], sk[3], sv[3];
  if (!prompt_rows(q, dev, sq) || !prompt_rows(k, dev, sk) || !prompt_rows(v, dev, sv)) Py_RETURN_NONE;
  const int64_t B = q.size(0), Hq = q.size(1), T = q.size(2), Hkv = k.size(1);
  if (k.size(0) != B || v.size(0) != B || v.size(1) != Hkv || k.size(2) != T || v.size(2) != T) Py_RETURN_NONE;
  const c10::OptionalDeviceGuard guard(dev);
  Tensor out = new_tensor({B, Hq, T, 128}, at::kHalf, dev);
  const int64_t so[3] = {Hq * T * 128, T * 128, 128};
  const int causal = a[4] == Py_True ? 1 : 0;
  const int rc = without_gil([&] {
    return api.hqekv_prompt_attn(q.data_ptr(), sq, k.data_ptr(), sk, v.data_ptr(), sv, out.data_ptr(), so, B, Hq, Hkv, T, 128, (float)scaling, causal,
                                 stream_of(dev));
  });
  if (rc) return raise_rc(rc, "prompt_attn");
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// prompt_last_rows(q, k, scaling, rows) -> (B, Hq, rows, T), the causal rule; None as above
PyObject *prompt_last_rows(PyObject *, PyObject *const *a, Py_ssize_t na) {
  HANDLE_TH_ERRORS
  if (na != 4) return PyErr_Format(PyExc_TypeError, "prompt_last_rows takes 4 arguments");
  if (!is_tensor(a[0]) || !is_tensor(a[1])) Py_RETURN_NONE;
  const Tensor &q = ten(a[0]), &k = ten(a[1]);
  const double scaling = PyFloat_AsDouble(a[2]);
  const int64_t rows = PyLong_AsLongLong(a[3]);
  if (PyErr_Occurred()) return nullptr;
  if (!q.is_cuda()) Py_RETURN_NONE;
  const at::Device dev = q.device();
  int64_t sq[3], sk[3];
  if (!prompt_rows(q, dev, sq) || !prompt_rows(k, dev, sk)) Py_RETURN_NONE;
  const int64_t B = q.size(0), Hq = q.size(1), T = q.size(2), Hkv = k.size(1);
  if (k.size(0) != B || k.size(2) != T || rows <= 0 || rows > T || rows > 32) Py_RETURN_NONE;
  const c10::OptionalDeviceGuard guard(dev);
  Tensor probs = new_tensor({B, Hq, rows, T}, at::kHalf, dev), ws;
  const int64_t need = api.hqekv_prompt_last_rows_workspace_bytes(B, Hq, T);
  if (need > 0) ws = new_tensor({need}, at::kByte, dev);
  const int rc = without_gil([&] {
    return api.hqekv_prompt_last_rows(q.data_ptr(), sq, k.data_ptr(), sk, nullptr, nullptr, probs.data_ptr(), B, Hq, Hkv, T, 128, rows, (float)scaling,
                                      need > 0 ? ws.data_ptr() : nullptr, need > 0 ? need : 0, stream_of(dev));
  });
  if (rc) return raise_rc(rc, "prompt_last_rows");
  return THPVariable_Wrap(probs);
  END_HANDLE_TH_ERRORS
}

// ------------------------------------------------------------------------------------------------ cache maintenance
// reconstruct(pkv, low_uniform, cover_fn) -> (K, V) dense, or None where the classes and the residual of a side do not
// name every position exactly once, or a field is not plain
PyObject *reconstruct(PyObject *, PyObject *const *a, Py_ssize_t na) {
  HANDLE_TH_ERRORS
  if (na != 3) return PyErr_Format(PyExc_TypeError, "reconstruct takes 3 arguments");
  PyObject *pkv = a[0];
  if (!PyTuple_Check(pkv) || PyTuple_GET_SIZE(pkv) != TUPLE_LEN || !PyLong_Check(PyTuple_GET_ITEM(pkv, TUPLE_LEN - 1))) Py_RETURN_NONE;
  const int64_t T = PyLong_AsLongLong(PyTuple_GET_ITEM(pkv, TUPLE_LEN - 1));
  const Tensor *some = nullptr;
  for (int i : {2, 8, 16, 24, 32, NEW_V})
    if (!some && is_tensor(PyTuple_GET_ITEM(pkv, i))) some = &ten(PyTuple_GET_ITEM(pkv, i));
  if (!some || !some->is_cuda() || some->dim() != 4) Py_RETURN_NONE;
  const at::Device dev = some->device();
  const int64_t B = some->size(0);
  Side k, v;
  const bool low_uniform = a[1] == Py_True;
  if (!read_side(pkv, true, low_uniform, B, dev, k) || !read_side(pkv, false, low_uniform, B, dev, v)) Py_RETURN_NONE;
  if (k.tokens != T || v.tokens != T || k.H != v.H || k.D != v.D || k.D % 32 || k.D > 4096) Py_RETURN_NONE;
  for (Side *s : {&k, &v}) {
    for (int i = 0; i < s->n; ++i)
      if (s->seg[i].bits == 16 && (uintptr_t)s->seg[i].data % 16) Py_RETURN_NONE;
    const int c = cover_once(s->idx, s->n_idx, s->class_tokens, a[2], false);
    if (c < 0) return nullptr;
    if (!c) Py_RETURN_NONE;
    if (s->tokens > s->class_tokens) s->seg[s->n - 1].pos_base = s->class_tokens;
  }
  const c10::OptionalDeviceGuard guard(dev);
  Tensor K = new_tensor({B, k.H, T, k.D}, at::kHalf, dev), V = new_tensor({B, k.H, T, k.D}, at::kHalf, dev);
  const int rc = without_gil(
      [&] { return api.hqekv_cache_reconstruct(k.seg, k.n, v.seg, v.n, K.data_ptr(), V.data_ptr(), B * k.H, k.D, T, stream_of(dev)); });
  if (rc) return raise_rc(rc, "cache_reconstruct");
  return Py_BuildValue("NN", THPVariable_Wrap(K), THPVariable_Wrap(V));
  END_HANDLE_TH_ERRORS
}

// importance(ring, n, total) -> (importance / 32 (total,), block scores (total / 32,)), or None
PyObject *importance(PyObject *, PyObject *const *a, Py_ssize_t na) {
  HANDLE_TH_ERRORS
  if (na != 3) return PyErr_Format(PyExc_TypeError, "importance takes 3 arguments");
  if (!is_tensor(a[0])) Py_RETURN_NONE;
  const Tensor &w = ten(a[0]);
  const int64_t n = PyLong_AsLongLong(a[1]), total = PyLong_AsLongLong(a[2]);
  if (PyErr_Occurred()) return nullptr;
  if (!w.is_cuda() || !plain_f16(w, 2, w.device()) || total <= 0 || total > n || total % 32) Py_RETURN_NONE;
  const at::Device dev = w.device();
  const c10::OptionalDeviceGuard guard(dev);
  Tensor imp = new_tensor({total}, at::kHalf, dev), scores = new_tensor({total / 32}, at::kHalf, dev);
  const int rc = without_gil([&] {
    return api.hqekv_importance_scores(w.data_ptr(), (int32_t)w.size(0), w.size(1), n, total, imp.data_ptr(), scores.data_ptr(), stream_of(dev));
  });
  if (rc) return raise_rc(rc, "importance_scores");
  return Py_BuildValue("NN", THPVariable_Wrap(imp), THPVariable_Wrap(scores));
  END_HANDLE_TH_ERRORS
}

// Block numbers of a position array that carries them (see cache_policy._host_blocks), written to `out` as int32.
bool known_blocks(PyObject *idx, std::vector<int32_t> &out) {
  const Tensor &t = ten(idx);
  PyObject *ver = PyObject_GetAttr(idx, s_host_version), *blocks = ver ? PyObject_GetAttr(idx, s_blocks) : nullptr;
  bool ok = false;
  if (ver && blocks && PyLong_Check(ver) && !t.is_inference() && PyLong_AsLongLong(ver) == (long long)t._version()) {
    Py_buffer b;
    if (PyObject_GetBuffer(blocks, &b, PyBUF_C_CONTIGUOUS | PyBUF_FORMAT) == 0) {
      if (b.itemsize == 8 && b.ndim == 1 && b.format && (b.format[0] == 'l' || b.format[0] == 'q') && b.len / 8 * 32 == t.numel()) {
        const int64_t *p = (const int64_t *)b.buf;
        out.assign(p, p + b.len / 8);
        ok = true;
      }
      PyBuffer_Release(&b);
    }
  }
  Py_XDECREF(ver);
  Py_XDECREF(blocks);
  if (PyErr_Occurred()) PyErr_Clear();
  return ok;
}

// One side's classes as sources of a migration, with their block numbers.
struct OldSide {
  hqekv_cache_class src[6] = {};
  std::vector<int32_t> blocks[5];
  int64_t n_blocks = 0;
};
constexpr int CLASS_BITS[5] = {16, 8, 4, 2, 1}, K_SLOT[5] = {0, 4, 12, 20, 28}, V_SLOT[5] = {2, 8, 16, 24, 32};

bool old_side(PyObject *pkv, bool is_k, bool low_normal, int64_t B, int64_t H, int64_t D, const at::Device &dev, OldSide &o) {
  for (int c = 0; c < 5; ++c) {
    const int slot = is_k ? K_SLOT[c] : V_SLOT[c], bits = CLASS_BITS[c];
    PyObject *data = PyTuple_GET_ITEM(pkv, slot), *idx = PyTuple_GET_ITEM(pkv, slot + 1);
    if (data == Py_None) continue;
    if (!is_tensor(data) || !is_tensor(idx)) return false;
    const Tensor &t = ten(data);
    hqekv_cache_class &e = o.src[c];
    if (bits == 16 ? !plain_f16(t, 4, dev) : !plain_i32(t, 4, dev)) return false;
    e.bits = bits;
    e.n_tokens = is_k ? t.size(3) * (bits == 16 ? 1 : 32 / bits) : t.size(2);
    if (t.size(0) != B || t.size(1) != H || (is_k ? t.size(2) : t.size(3) * (bits == 16 ? 1 : 32 / bits)) != D || ten(idx).numel() != e.n_tokens)
      return false;
    e.data = t.data_ptr();
    if (bits != 16) {
      PyObject *sc = PyTuple_GET_ITEM(pkv, slot + 2), *zr = PyTuple_GET_ITEM(pkv, slot + 3);
      if (!is_tensor(sc) || !is_tensor(zr) || !plain_f16(ten(sc), 4, dev) || !plain_f16(ten(zr), 4, dev)) return false;
      e.scale = ten(sc).data_ptr();
      e.zero = ten(zr).data_ptr();
      if (bits == 1 && low_normal) e.layout = HQEKV_LAYOUT_NORMAL1;
    }
    if (!known_blocks(idx, o.blocks[c])) return false;
    o.n_blocks += (int64_t)o.blocks[c].size();
  }
  return true;
}

// A tensor over a part of another's storage, without the dispatcher's way of making a view (two dozen of them per
// compression).
Tensor part_of(const Tensor &base, at::IntArrayRef shape, int64_t offset) {
  Tensor t = at::detail::make_tensor<c10::TensorImpl>(c10::Storage(base.storage()), base.key_set(), base.dtype());
  t.unsafeGetTensorImpl()->set_sizes_contiguous(shape);
  t.unsafeGetTensorImpl()->set_storage_offset(offset);
  return t;
}

int64_t up(int64_t n, int64_t a) { return (n + a - 1) / a * a; }

// The new classes of one side: three allocations, tensors over parts of them.
struct NewSide {
  hqekv_cache_class dst[5] = {};
  Tensor data[5], scale[5], zero[5], idx[5];
  int n_dst = 0;
};

void new_side(bool is_k, bool low_normal, const int32_t *counts, int64_t B, int64_t H, int64_t D, const at::Device &dev, NewSide &o) {
  int64_t n16 = 0, n32 = 0, n64 = 0;
  struct {
    int64_t n, o_data, o_scale, o_zero, o_idx;
  } at_[5];
  for (int c = 0; c < 5; ++c) {
    const int bits = CLASS_BITS[c];
    const int64_t n = (int64_t)counts[c] * 32;
    auto &p = at_[c];
    p.n = n;
    if (!n) continue;
    if (bits == 16) {
      p.o_data = n16;
      n16 += up(B * H * D * n, 128);
    } else {
      const int64_t groups = up(B * H * n * D / 32, 128);
      p.o_scale = n16;
      p.o_zero = n16 + groups;
      n16 += 2 * groups;
      p.o_data = n32;
      n32 += up(B * H * D * n * bits / 32, 64);
    }
    p.o_idx = n64;
    n64 += n;
  }
  if (!n64) return;
  const Tensor b16 = new_tensor({std::max<int64_t>(n16, 1)}, at::kHalf, dev), b32 = new_tensor({std::max<int64_t>(n32, 1)}, at::kInt, dev),
               b64 = new_tensor({n64}, at::kLong, dev);
  for (int c = 0; c < 5; ++c) {
    const auto &p = at_[c];
    if (!p.n) continue;
    const int bits = CLASS_BITS[c];
    hqekv_cache_class &e = o.dst[o.n_dst++];
    e.bits = bits;
    e.n_tokens = p.n;
    o.idx[c] = part_of(b64, {p.n}, p.o_idx);
    e.idx = (int64_t *)o.idx[c].data_ptr();
    if (bits == 16) {
      o.data[c] = is_k ? part_of(b16, {B, H, D, p.n}, p.o_data) : part_of(b16, {B, H, p.n, D}, p.o_data);
    } else {
      o.data[c] = is_k ? part_of(b32, {B, H, D, p.n * bits / 32}, p.o_data) : part_of(b32, {B, H, p.n, D * bits / 32}, p.o_data);
      const int64_t shape[4] = {B, H, is_k ? D : p.n, (is_k ? p.n : D) / 32};
      o.scale[c] = part_of(b16, shape, p.o_scale);
      o.zero[c] = part_of(b16, shape, p.o_zero);
      e.scale = o.scale[c].data_ptr();
      e.zero = o.zero[c].data_ptr();
      if (bits == 1 && low_normal) e.layout = HQEKV_LAYOUT_NORMAL1;
    }
    e.data = o.data[c].data_ptr();
  }
}

void put_item(PyObject *tuple, int i, PyObject *v) {
  PyObject *old = PyTuple_GET_ITEM(tuple, i);
  PyTuple_SET_ITEM(tuple, i, v);
  Py_XDECREF(old);
}

// The fields of one side into the new tuple.  The kernel writes the positions behind torch's back, and what rides on
// the arrays says exactly what it writes: the block numbers (positions: numpy int64, class after class), for the next
// compression, and -- the classes together are a permutation of the n_blocks surviving blocks -- the verdict of
// attention.idx_cover_once about these arrays: every position once, in whole runs of 32.
bool put_side(PyObject *tuple, bool is_k, const NewSide &o, const int32_t *counts, int64_t n_blocks, PyObject *positions, PyObject *weak_ref) {
  PyObject *idx[5];
  int n_idx = 0;
  int64_t blk = 0;
  for (int c = 0; c < 5; ++c) {
    if (!counts[c]) continue;
    const int slot = is_k ? K_SLOT[c] : V_SLOT[c];
    put_item(tuple, slot, THPVariable_Wrap(o.data[c]));
    if (CLASS_BITS[c] != 16) {
      put_item(tuple, slot + 2, THPVariable_Wrap(o.scale[c]));
      put_item(tuple, slot + 3, THPVariable_Wrap(o.zero[c]));
    }
    PyObject *i = idx[n_idx++] = THPVariable_Wrap(o.idx[c]);
    put_item(tuple, slot + 1, i);
    PyObject *mine = PySequence_GetSlice(positions, blk, blk + counts[c]), *ver = PyLong_FromLongLong((long long)o.idx[c]._version());
    const bool ok = mine && ver && PyObject_SetAttr(i, s_blocks, mine) == 0 && PyObject_SetAttr(i, s_host_version, ver) == 0;
    Py_XDECREF(mine);
    Py_XDECREF(ver);
    if (!ok) return false;
    blk += counts[c];
  }
  if (!n_idx) return true;
  PyObject *key = PyTuple_New(n_idx + 1), *refs = PyList_New(n_idx);
  bool ok = key && refs;
  for (int i = 0; ok && i < n_idx; ++i) {
    const Tensor &t = ten(idx[i]);
    PyObject *k = Py_BuildValue("KLL", (unsigned long long)(uintptr_t)t.data_ptr(), (long long)t.numel(), (long long)t._version());
    PyObject *r = PyObject_CallFunctionObjArgs(weak_ref, idx[i], nullptr);
    ok = k && r;
    PyTuple_SET_ITEM(key, i, k);
    PyList_SET_ITEM(refs, i, r);
  }
  if (ok) {
    PyTuple_SET_ITEM(key, n_idx, PyLong_FromLongLong((long long)n_blocks * 32));
    PyObject *cover = Py_BuildValue("(OOOO)", key, Py_True, refs, Py_True);
    ok = cover && PyObject_SetAttr(idx[0], s_cover, cover) == 0;
    Py_XDECREF(cover);
  }
  Py_XDECREF(key);
  Py_XDECREF(refs);
  return ok;
}

bool new_tokens(const Tensor &t, bool is_k, int64_t B, int64_t H, int64_t n, int64_t D, const at::Device &dev, hqekv_cache_class &e) {
  if (t.dim() != 4 || t.scalar_type() != at::kHalf || t.device() != dev || t.size(0) != B || t.size(1) != H || t.size(2) < n || t.size(3) != D ||
      t.stride(3) != 1 || t.stride(2) != D || ((H > 1 || B > 1) && (t.stride(1) % D || t.stride(1) < n * D)) || (B > 1 && t.stride(0) != H * t.stride(1)))
    return false;
  e.bits = 16;
  e.n_tokens = n;
  e.data = t.data_ptr();
  e.slab_tokens = H > 1 || B > 1 ? t.stride(1) / D : n;
  e.layout = is_k ? HQEKV_LAYOUT_TOKEN_MAJOR : 0;
  return true;
}

// Both block rankings, written by one launch into page-locked memory.  Every entry is stored exactly once, so the ranking
// is there as soon as no entry holds its initial value: that is watched, closely at first (a stream synchronisation wakes up
// some ten microseconds later), then, where a model's work is queued ahead, every 20 us until the stream has nothing left to do.
// The stream is not waited for: what is queued behind the ranking would be waited for as well.  meanwhile: None, or what the
// caller has to queue that does not need the ranking -- the kernels run it while the host reads the ranking and plans; called
// once, behind the launch.  (The memory may not be let go before the kernel has written it: what the call raises is raised
// after the wait.)
bool host_orders(const void *const (&scores)[2], int64_t n, const Tensor &order, const at::Device &dev, PyObject *meanwhile) {
  volatile int32_t *p = (volatile int32_t *)order.data_ptr();
  for (int64_t i = 0; i < 2 * n; ++i) p[i] = -1;
  hipError_t err = hipSuccess;
  auto wait = [&] {
    const auto until = std::chrono::steady_clock::now() + std::chrono::milliseconds(2);
    int64_t i = 0;
    while (i < 2 * n) {
      if (p[i] >= 0) {
        ++i;
      } else if (std::chrono::steady_clock::now() > until) {
        err = hipStreamQuery((hipStream_t)stream_of(dev));
        if (err != hipErrorNotReady) break;
        err = hipSuccess;
        (void)hipGetLastError();   // (an answer, not an error for the next launch to find)
        std::this_thread::sleep_for(std::chrono::microseconds(20));
      }
    }
    return HQEKV_OK;
  };
  const int rc = without_gil([&]() -> int {
    const int rc = api.hqekv_rank_blocks(scores, 2, n, (int32_t *)order.data_ptr(), stream_of(dev));
    return rc || meanwhile != Py_None ? rc : wait();
  });
  if (rc) {
    raise_rc(rc, "rank_blocks");
    return false;
  }
  bool raised = false;
  if (meanwhile != Py_None) {
    PyObject *did = PyObject_CallNoArgs(meanwhile);
    raised = !did;
    Py_XDECREF(did);
    without_gil(wait);
  }
  if (raised) return false;
  if (err != hipSuccess) PyErr_Format(PyExc_RuntimeError, "rank_blocks: HIP error %d", (int)err);
  return err == hipSuccess;
}

bool six_counts(PyObject *o, int64_t (&out)[6], int &n) {
  if (!is_tensor(o)) return false;
  const Tensor &t = ten(o);
  if (!t.device().is_cpu() || t.dim() != 1 || !t.is_contiguous() || (t.numel() != 5 && t.numel() != 6)) return false;
  n = (int)t.numel();
  if (t.scalar_type() == at::kInt)
    for (int i = 0; i < n; ++i) out[i] = t.data_ptr<int32_t>()[i];
  else if (t.scalar_type() == at::kLong)
    for (int i = 0; i < n; ++i) out[i] = t.data_ptr<int64_t>()[i];
  else return false;
  return true;
}

// compress(pkv, history, length, k_scores, importance, times_range, V_range or None, K_counts, V_counts, low_normal,
// ring or None, (K buffer, V buffer) or None, new_array, weak_ref[, meanwhile or None]): cache_policy.compress for a cache,
// rankings and counts made of whole blocks.  ring: the importance ring, whose evicted columns are taken out; buffers (B, H,
// capacity, D): where the residual goes, its fields are their heads then.  new_array(n): an int64 numpy array; weak_ref:
// weakref.ref; meanwhile(): see host_orders -- not called where None is returned before the ranking is launched.
// -> (the new tuple, positions kept where tokens were evicted and no ring was given, else None), or None where that does not
// hold -- found out before anything is launched except the score and rank kernels.
PyObject *compress(PyObject *, PyObject *const *a, Py_ssize_t na) {
  HANDLE_TH_ERRORS
  if (na != 14 && na != 15) return PyErr_Format(PyExc_TypeError, "compress takes 14 or 15 arguments");
  PyObject *pkv = a[0];
  const int64_t history = PyLong_AsLongLong(a[1]), length = PyLong_AsLongLong(a[2]);
  if (PyErr_Occurred()) return nullptr;
  const bool times_range = a[5] == Py_True, low_normal = a[9] == Py_True;
  if (!PyTuple_Check(pkv) || PyTuple_GET_SIZE(pkv) != TUPLE_LEN || !is_tensor(a[3]) || !is_tensor(a[4])) Py_RETURN_NONE;
  PyObject *nk = PyTuple_GET_ITEM(pkv, NEW_K), *nv = PyTuple_GET_ITEM(pkv, NEW_V), *prev = PyTuple_GET_ITEM(pkv, RANGES);
  if (!is_tensor(nk) || !is_tensor(nv)) Py_RETURN_NONE;
  const Tensor &newK = ten(nk), &newV = ten(nv), &scores_k = ten(a[3]), &imp = ten(a[4]);
  if (!newV.is_cuda() || newV.dim() != 4) Py_RETURN_NONE;
  const at::Device dev = newV.device();
  const int64_t B = newV.size(0), H = newV.size(1), D = newV.size(3), total = history + length, nb = total / 32;
  if (total <= 0 || total % 32 || history % 32 || length <= 0 || nb > 32768 || D % 32 || B * H > 1024) Py_RETURN_NONE;
  if (!plain_f16(imp, 1, dev) || imp.numel() != total || !plain_f16(scores_k, 1, dev) || scores_k.numel() != nb) Py_RETURN_NONE;
  OldSide ks, vs;
  int64_t kc[6] = {}, vc[6] = {};
  int n_k = 0, n_v = 0;
  if (!six_counts(a[7], kc, n_k) || !six_counts(a[8], vc, n_v) || !new_tokens(newK, true, B, H, length, D, dev, ks.src[5]) ||
      !new_tokens(newV, false, B, H, length, D, dev, vs.src[5]) || !old_side(pkv, true, low_normal, B, H, D, dev, ks) ||
      !old_side(pkv, false, low_normal, B, H, D, dev, vs) || ks.n_blocks != history / 32 || vs.n_blocks != history / 32)
    Py_RETURN_NONE;
  if (((uintptr_t)newV.data_ptr() | (uintptr_t)newK.data_ptr()) % 16) Py_RETURN_NONE;
  for (const int64_t *c : {kc, vc}) {   // what the planner will ask for
    int64_t sum = 0;
    for (int i = 0; i < 6; ++i) {
      if (c[i] < 0 || c[i] % 32) Py_RETURN_NONE;
      sum += c[i];
    }
    if (sum != total) Py_RETURN_NONE;
  }
  hqekv_migrate_extra x{};
  Tensor ring;
  if (a[10] != Py_None) {
    if (!is_tensor(a[10])) Py_RETURN_NONE;
    ring = ten(a[10]);
    if (!plain_f16(ring, 2, dev) || ring.size(1) < total || ring.size(0) > 65535) Py_RETURN_NONE;
  }
  const int64_t rk = newK.size(2) - length, rv = newV.size(2) - length;
  if (rk != rv) Py_RETURN_NONE;
  Tensor resK, resV;
  if (rk) {
    if (a[11] != Py_None) {
      if (!PyTuple_Check(a[11]) || PyTuple_GET_SIZE(a[11]) != 2 || !is_tensor(PyTuple_GET_ITEM(a[11], 0)) || !is_tensor(PyTuple_GET_ITEM(a[11], 1))) Py_RETURN_NONE;
      resK = ten(PyTuple_GET_ITEM(a[11], 0));
      resV = ten(PyTuple_GET_ITEM(a[11], 1));
      for (const Tensor *t : {&resK, &resV})
        if (!plain_f16(*t, 4, dev) || t->size(0) != B || t->size(1) != H || t->size(2) < rk || t->size(3) != D) Py_RETURN_NONE;
    } else {
      resK = new_tensor({B, H, rk, D}, at::kHalf, dev);
      resV = new_tensor({B, H, rv, D}, at::kHalf, dev);
    }
  }
  const c10::OptionalDeviceGuard guard(dev);
  void *stream = stream_of(dev);
  // ---- token ranges of V -- the older ones and the new tokens' -- and the scores of the V side's blocks
  Tensor range;
  const Tensor scores_v = new_tensor({nb}, at::kHalf, dev);
  int rc = 0;
  if (a[6] != Py_None) {
    if (!is_tensor(a[6])) Py_RETURN_NONE;
    range = ten(a[6]);
    if (!plain_f16(range, 1, dev) || range.numel() != total) Py_RETURN_NONE;
    rc = without_gil(
        [&] { return api.hqekv_weighted_block_scores(imp.data_ptr(), times_range ? range.data_ptr() : nullptr, total, scores_v.data_ptr(), stream); });
  } else {
    if (prev == Py_None ? history != 0 : (!is_tensor(prev) || !plain_f16(ten(prev), 1, dev) || ten(prev).numel() != history)) Py_RETURN_NONE;
    range = new_tensor({total}, at::kHalf, dev);
    const void *older = history ? ten(prev).data_ptr() : nullptr;
    rc = without_gil([&] {
      return api.hqekv_range_block_scores(newV.data_ptr(), B, H, length, D, vs.src[5].slab_tokens, older, history, imp.data_ptr(), times_range ? 1 : 0,
                                          range.data_ptr(), scores_v.data_ptr(), stream);
    });
  }
  if (rc) return raise_rc(rc, "range_block_scores");
  // ---- both rankings
  const Tensor host = at::empty({2 * nb + 5 * nb + 4}, at::TensorOptions().dtype(at::kInt).pinned_memory(true));
  const void *const sc[2] = {scores_k.data_ptr(), scores_v.data_ptr()};
  const Tensor up_d = new_tensor({5 * nb}, at::kInt, dev);   // (made while the ranking runs)
  if (!host_orders(sc, nb, host, dev, na > 14 ? a[14] : Py_None)) return nullptr;
  // ---- the plans of both sides and the V side's surviving blocks, one transfer for all
  const int32_t *order = (const int32_t *)host.data_ptr();
  int32_t *words = (int32_t *)host.data_ptr() + up(2 * nb, 4), counts[2][5] = {}, n_alive[2] = {0, 0};
  std::vector<int64_t> order64(nb);
  std::vector<int32_t> alive_k(nb);
  for (int side = 0; side < 2; ++side) {
    OldSide &o = side ? vs : ks;
    const int32_t *old[5];
    int32_t cnt[5];
    for (int c = 0; c < 5; ++c) {
      old[c] = o.blocks[c].data();
      cnt[c] = (int32_t)o.blocks[c].size();
    }
    for (int64_t i = 0; i < nb; ++i) order64[i] = order[side * nb + i];
    rc = without_gil([&] {
      return api.hqekv_plan_side(old, cnt, (int32_t)(history / 32), (int32_t)(length / 32), order64.data(), side ? vc : kc, side ? n_v : n_k, counts[side],
                                 words + side * 2 * nb, side ? words + 4 * nb : alive_k.data(), &n_alive[side]);
    });
    if (rc) Py_RETURN_NONE;   // not a whole-block selection after all
  }
  const bool evicted = n_alive[1] < nb;
  rc = without_gil([&] { return api.hqekv_fetch_words(words, up_d.data_ptr(), evicted ? 4 * nb + n_alive[1] : 4 * nb, stream); });
  if (rc) return raise_rc(rc, "fetch_words");
  at::getHostAllocator(at::kCUDA)->record_event(host.data_ptr(), host.storage().data_ptr().get_context(),
                                                c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(dev.index()).unwrap());
  // ---- the launch that moves everything
  NewSide k_new, v_new;
  new_side(true, low_normal, counts[0], B, H, D, dev, k_new);
  new_side(false, low_normal, counts[1], B, H, D, dev, v_new);
  const int32_t *plan = (const int32_t *)up_d.data_ptr();
  Tensor kept_range = range;
  if (evicted) {
    const int32_t *alive = words + 4 * nb;
    x.alive = plan + 4 * nb;
    x.n_alive = n_alive[1];
    while (x.first_moved < x.n_alive && alive[x.first_moved] == x.first_moved) ++x.first_moved;
    if (ring.defined()) {
      x.ring = ring.data_ptr();
      x.ring_rows = (int32_t)ring.size(0);
      x.ring_stride = ring.size(1);
    }
    kept_range = new_tensor({32 * (int64_t)n_alive[1]}, at::kHalf, dev);
    x.range_in = range.data_ptr();
    x.range_out = kept_range.data_ptr();
  }
  if (rk) {
    const Tensor *src[2] = {&newK, &newV}, *dst[2] = {&resK, &resV};
    x.res_rows = (int32_t)rk;
    for (int side = 0; side < 2; ++side) {
      x.res_src[side] = (const char *)src[side]->data_ptr() + 2 * D * length;
      x.res_src_slab[side] = (side ? vs : ks).src[5].slab_tokens;
      x.res_dst[side] = dst[side]->data_ptr();
      x.res_dst_slab[side] = dst[side]->size(2);
    }
  }
  rc = without_gil([&] {
    return api.hqekv_cache_migrate_both(ks.src, 6, k_new.dst, k_new.n_dst, plan, vs.src, 6, v_new.dst, v_new.n_dst, plan + 2 * nb, B * H, D, &x, stream);
  });
  if (rc) return raise_rc(rc, "cache_migrate");
  // ---- the new tuple, while it runs
  PyObject *out = PyTuple_New(TUPLE_LEN);
  if (!out) return nullptr;
  for (int i = 0; i < TUPLE_LEN; ++i) {
    PyObject *o = (i < 36 || i == RANGES || i == NEW_K || i == NEW_V) ? Py_None : PyTuple_GET_ITEM(pkv, i);
    Py_INCREF(o);
    PyTuple_SET_ITEM(out, i, o);
  }
  for (int side = 0; side < 2; ++side) {
    PyObject *pos = PyObject_CallFunction(a[12], "L", (long long)n_alive[side]);
    Py_buffer b;
    if (!pos || PyObject_GetBuffer(pos, &b, PyBUF_WRITABLE | PyBUF_C_CONTIGUOUS) != 0) {
      Py_XDECREF(pos);
      Py_DECREF(out);
      return nullptr;
    }
    const int32_t *w = words + side * 2 * nb;
    const bool room = b.len == 8 * (Py_ssize_t)n_alive[side];
    for (int32_t i = 0; room && i < n_alive[side]; ++i) ((int64_t *)b.buf)[i] = w[n_alive[side] + i];
    PyBuffer_Release(&b);
    const bool ok = room && put_side(out, side == 0, side ? v_new : k_new, counts[side], n_alive[side], pos, a[13]);
    Py_DECREF(pos);
    if (!ok) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "new_array");
      Py_DECREF(out);
      return nullptr;
    }
  }
  put_item(out, RANGES, THPVariable_Wrap(kept_range));
  if (rk) {
    put_item(out, NEW_K, THPVariable_Wrap(resK.size(2) > rk ? rows_of(resK, 0, rk) : resK));
    put_item(out, NEW_V, THPVariable_Wrap(resV.size(2) > rk ? rows_of(resV, 0, rk) : resV));
  }
  if (!evicted || ring.defined()) return Py_BuildValue("NO", out, Py_None);
  Tensor keep = at::empty({32 * (int64_t)n_alive[1]}, at::TensorOptions().dtype(at::kLong));
  int64_t *p = (int64_t *)keep.data_ptr();
  for (int32_t i = 0; i < n_alive[1]; ++i)
    for (int j = 0; j < 32; ++j) *p++ = (int64_t)words[4 * nb + i] * 32 + j;
  return Py_BuildValue("NN", out, THPVariable_Wrap(keep.to(dev)));
  END_HANDLE_TH_ERRORS
}

// bind(path): take the kernels' entry points from this library
PyObject *bind(PyObject *, PyObject *path) {
  const char *p = PyUnicode_AsUTF8(path);
  if (!p) return nullptr;
  void *h = dlopen(p, RTLD_NOW | RTLD_LOCAL);
  if (!h) return PyErr_Format(PyExc_RuntimeError, "%s", dlerror());
#define X(n_)                                     \
  api.n_ = (decltype(&::n_))dlsym(h, #n_);        \
  if (!api.n_) return PyErr_Format(PyExc_RuntimeError, "%s lacks %s", p, #n_);
  HQ_SYMBOLS(X)
#undef X
  Py_RETURN_NONE;
}

PyMethodDef module_methods[] = {
    {"bind", bind, METH_O, nullptr},
    {"decode", (PyCFunction)(void (*)(void))decode, METH_FASTCALL, nullptr},
    {"step_tables", (PyCFunction)(void (*)(void))step_tables, METH_FASTCALL, nullptr},
    {"prompt_attention", (PyCFunction)(void (*)(void))prompt_attention, METH_FASTCALL, nullptr},
    {"prompt_last_rows", (PyCFunction)(void (*)(void))prompt_last_rows, METH_FASTCALL, nullptr},
    {"reconstruct", (PyCFunction)(void (*)(void))reconstruct, METH_FASTCALL, nullptr},
    {"importance", (PyCFunction)(void (*)(void))importance, METH_FASTCALL, nullptr},
    {"compress", (PyCFunction)(void (*)(void))compress, METH_FASTCALL, nullptr},
    {"quantize_into", (PyCFunction)(void (*)(void))quantize_into, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, module_methods};

bool add_type(PyObject *m, PyTypeObject &t, const char *qualified, const char *name, size_t size, newfunc make, destructor free_,
              PyMethodDef *methods, PyGetSetDef *fields, unsigned long flags) {
  t.tp_name = qualified;
  t.tp_basicsize = (Py_ssize_t)size;
  t.tp_flags = Py_TPFLAGS_DEFAULT | flags;
  t.tp_new = make;
  t.tp_dealloc = free_;
  t.tp_methods = methods;
  t.tp_getset = fields;
  if (PyType_Ready(&t) < 0) return false;
  Py_INCREF(&t);
  return PyModule_AddObject(m, name, (PyObject *)&t) == 0;
}

}  // namespace

PyMODINIT_FUNC PyInit__host(void) {
  PyObject *m = PyModule_Create(&module_def);
  if (!m) return nullptr;
  s_cover = PyUnicode_InternFromString("_hq_cover");
  s_blocks = PyUnicode_InternFromString("_hq_blocks");
  s_host_version = PyUnicode_InternFromString("_hq_host_version");
  if (!s_cover || !s_blocks || !s_host_version ||
      !add_type(m, tables_type, "hqekv_amd._host.StepTables", "StepTables", sizeof(StepTables), tables_new, tables_free, tables_methods,
                nullptr, 0) ||
      !add_type(m, kivi_type, "hqekv_amd._host.KiviState", "KiviState", sizeof(KiviState), kivi_new, kivi_free, kivi_methods, kivi_fields, 0)) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
