// Native launch path of the Python operators: one CPython call that reads the
// tensors' addresses, shapes and strides, checks them, allocates the outputs
// and calls the C ABI on torch's current stream.
//
// Each function handles the common form of a call (plain strided GPU tensors
// that pass every check) and returns None for anything else, having done
// nothing; the caller in ops.py then runs its own checks, which raise the
// precise error or take the general path.  So these decide no error and refuse
// nothing.
//
// Why: the same work in Python (tensor attribute reads, reshapes and a ctypes
// call of 13 to 40 converted arguments) took about 18 us an operator, longer
// than most launches run: the four launches of an 8B layer at 61 tokens were
// 10 us of GPU time in 75 us.
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ops/empty.h>
#include <c10/hip/HIPStream.h>

#include "../../include/my_vllm_amd.h"

namespace {

using at::Tensor;

constexpr int kHeadDim = 128;

// A plain strided GPU tensor (no subclass, no functorch or functionalization
// wrapper), or nullptr.
const Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const Tensor& t = THPVariable_Unpack(o);
  static const c10::DispatchKeySet wrapped(
      {c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
       c10::DispatchKey::Functionalize, c10::DispatchKey::ZeroTensor, c10::DispatchKey::Conjugate,
       c10::DispatchKey::Negative});
  if (!t.defined() || !t.is_cuda() || t.layout() != c10::kStrided || t.key_set().has_any(wrapped)) return nullptr;
  return &t;
}

int dtype_code(const Tensor& t) {
  if (t.scalar_type() == at::kBFloat16) return MVA_DTYPE_BF16;
  if (t.scalar_type() == at::kHalf) return MVA_DTYPE_F16;
  return -1;
}

// MVA_DTYPE_* of norm weights for activations of x's type, or -1.
int weight_code(const Tensor& w, const Tensor& x) {
  if (w.scalar_type() == x.scalar_type()) return dtype_code(x);
  return w.scalar_type() == at::kFloat ? MVA_DTYPE_F32 : -1;
}

void* stream_of(const Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

void* ptr(const Tensor& t) { return t.data_ptr(); }

PyObject* none() { Py_RETURN_NONE; }

// The status of `launch`, run without the GIL, as a ctypes call runs it: a
// launch that waits for room in a full queue stops no other Python thread, and
// none that a host callback in the queue waits for.  The arguments are read
// before it is released.
template <typename... P, typename... A>
int unlocked(int (*launch)(P...), A... args) {
  struct Released {
    PyThreadState* const state = PyEval_SaveThread();
    ~Released() { PyEval_RestoreThread(state); }
  } released;
  return launch(args...);
}

// `result` (a new reference) when the launch went out, else its error.
PyObject* launched(const char* name, int status, PyObject* result) {
  if (status == 0) return result;
  Py_XDECREF(result);
  return PyErr_Format(PyExc_RuntimeError, "%s failed (%d): %s", name, status, mva_last_error());
}
PyObject* launched(const char* name, int status) {
  Py_INCREF(Py_True);
  return launched(name, status, Py_True);
}
PyObject* launched(const char* name, int status, const Tensor& out) {
  return launched(name, status, status == 0 ? THPVariable_Wrap(out) : nullptr);
}

// Integer and float arguments; false (no Python error left) when one is not.
bool as_int(PyObject* o, int64_t* v) {
  if (!PyLong_Check(o)) return false;
  *v = PyLong_AsLongLong(o);
  if (*v == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}
bool as_float(PyObject* o, double* v) {
  if (!PyFloat_Check(o)) return false;
  *v = PyFloat_AS_DOUBLE(o);
  return true;
}

// Rows of the last dimension at one row stride: 2-D with unit inner stride,
// or contiguous.  Returns the row count, or -1.
int64_t row_view(const Tensor& t, int64_t hidden, int64_t* stride) {
  if (t.dim() == 2 && t.stride(1) == 1) {
    *stride = t.size(0) > 1 ? t.stride(0) : hidden;
    return t.size(0);
  }
  if (t.dim() > 2 && t.is_contiguous()) {
    *stride = hidden;
    return t.numel() / hidden;
  }
  return -1;
}

// Runs `body` and turns a C++ exception into "not handled".
template <typename F>
PyObject* guarded(F body) {
  try {
    return body();
  } catch (const std::exception&) {
    PyErr_Clear();
    return none();
  }
}

PyObject* silu_and_mul(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    const Tensor* x = n == 1 ? plain(a[0]) : nullptr;
    if (!x || !x->is_contiguous() || x->dim() < 1 || x->numel() == 0) return none();
    const int code = dtype_code(*x);
    const int64_t width = x->size(-1);
    if (code < 0 || width % 2) return none();
    c10::SmallVector<int64_t, 5> shape(x->sizes().begin(), x->sizes().end());
    shape.back() = width / 2;
    const Tensor out = at::empty(shape, x->options().requires_grad(false));
    void* const stream = stream_of(*x);
    const int status = unlocked(mva_silu_and_mul, ptr(*x), ptr(out), x->numel() / width, width / 2, code, stream);
    return launched("mva_silu_and_mul", status, out);
  });
}

// (x, weight, eps): contiguous rows or a [tokens, heads, hidden] view.
PyObject* rms_norm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    double eps;
    if (n != 3 || !as_float(a[2], &eps)) return none();
    const Tensor *x = plain(a[0]), *w = plain(a[1]);
    if (!x || !w || x->device() != w->device() || !w->is_contiguous()) return none();
    const int code = dtype_code(*x), wcode = weight_code(*w, *x);
    const int64_t hidden = w->numel();
    if (code < 0 || wcode < 0 || x->dim() < 2 || x->dim() > 3 || x->numel() == 0 || x->size(-1) != hidden ||
        x->stride(-1) != 1)
      return none();
    const bool heads = x->dim() == 3;
    const int64_t per_group = heads ? x->size(1) : 1;
    const int64_t rows = x->size(0) * per_group;
    const int64_t row_stride = heads ? x->stride(1) : x->size(0) > 1 ? x->stride(0) : hidden;
    const int64_t group_stride = heads ? x->stride(0) : row_stride;
    const Tensor out = at::empty(x->sizes(), x->options().requires_grad(false));
    void* const stream = stream_of(*x);
    const int status = unlocked(
        mva_rms_norm, ptr(*x), group_stride, row_stride, ptr(*w), ptr(out), per_group * hidden, hidden, rows,
        per_group, hidden, (float)eps, code, wcode, stream);
    return launched("mva_rms_norm", status, out);
  });
}

// (x, residual, weight, eps, inplace)
PyObject* fused_add_rms_norm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    double eps;
    if (n != 5 || !as_float(a[3], &eps) || !PyBool_Check(a[4])) return none();
    const bool inplace = a[4] == Py_True;
    const Tensor *x = plain(a[0]), *r = plain(a[1]), *w = plain(a[2]);
    if (!x || !r || !w || x->device() != r->device() || x->device() != w->device() || !w->is_contiguous()) return none();
    const int code = dtype_code(*x), wcode = weight_code(*w, *x);
    const int64_t hidden = w->numel();
    if (code < 0 || wcode < 0 || r->scalar_type() != x->scalar_type() || x->dim() < 2 || x->numel() == 0 ||
        x->size(-1) != hidden || x->sizes() != r->sizes())
      return none();
    int64_t xs, rs;
    const int64_t rows = row_view(*x, hidden, &xs);
    if (rows < 0 || row_view(*r, hidden, &rs) < 0) return none();
    const auto options = x->options().requires_grad(false);
    const Tensor out = inplace ? *x : at::empty(x->sizes(), options);
    const Tensor res = inplace ? *r : at::empty(x->sizes(), options);
    void* const stream = stream_of(*x);
    const int status = unlocked(
        mva_fused_add_rms_norm, ptr(*x), xs, ptr(*r), rs, ptr(*w), ptr(out), inplace ? xs : hidden, ptr(res),
        inplace ? rs : hidden, rows, hidden, (float)eps, code, wcode, stream);
    if (status != 0) return launched("mva_fused_add_rms_norm", status, nullptr);
    if (inplace) return PyTuple_Pack(2, a[0], a[1]);
    PyObject* pair = PyTuple_New(2);
    if (pair == nullptr) return nullptr;
    PyTuple_SET_ITEM(pair, 0, THPVariable_Wrap(out));
    PyTuple_SET_ITEM(pair, 1, THPVariable_Wrap(res));
    return pair;
  });
}

bool head_rows(const Tensor& t, const Tensor& like) {
  return t.dim() == 3 && t.size(2) == kHeadDim && t.stride(2) == 1 && t.scalar_type() == like.scalar_type() &&
         t.device() == like.device();
}

bool slot_list(const Tensor& t, const Tensor& like, int64_t tokens) {
  return (t.scalar_type() == at::kInt || t.scalar_type() == at::kLong) && t.device() == like.device() &&
         t.dim() == 1 && t.numel() == tokens && t.is_contiguous();
}

// (positions, q, k, table, wq | None, wk | None, eps, v, k_cache, v_cache,
//  slots, q_out, k_out); with a store only.  True when launched.
PyObject* qk_norm_rope_store(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    double eps;
    if (n != 13 || !as_float(a[6], &eps)) return none();
    const Tensor *pos = plain(a[0]), *q = plain(a[1]), *k = plain(a[2]), *table = plain(a[3]);
    const Tensor *v = plain(a[7]), *kc = plain(a[8]), *vc = plain(a[9]), *slots = plain(a[10]);
    const Tensor *qo = plain(a[11]), *ko = plain(a[12]);
    const bool norm = a[4] != Py_None;
    const Tensor *wq = norm ? plain(a[4]) : nullptr, *wk = norm ? plain(a[5]) : nullptr;
    if (!pos || !q || !k || !table || !v || !kc || !vc || !slots || !qo || !ko || (norm && (!wq || !wk)) ||
        (!norm && a[5] != Py_None))
      return none();
    const int code = dtype_code(*q);
    const int64_t tokens = q->dim() == 3 ? q->size(0) : 0;
    if (code < 0 || tokens == 0 || !head_rows(*q, *q) || !head_rows(*k, *q) || !head_rows(*v, *q)) return none();
    if (k->size(0) != tokens || v->size(0) != tokens || v->size(1) != k->size(1)) return none();
    if (pos->scalar_type() != at::kLong || pos->dim() != 1 || pos->size(0) != tokens || !pos->is_contiguous() ||
        pos->device() != q->device())
      return none();
    if (table->scalar_type() != at::kFloat || !table->is_contiguous() || table->device() != q->device() ||
        table->dim() < 1 || table->size(0) == 0 || table->numel() != table->size(0) * kHeadDim)
      return none();
    if (qo->sizes() != q->sizes() || qo->strides() != q->strides() || ko->sizes() != k->sizes() ||
        ko->strides() != k->strides() || !head_rows(*qo, *q) || !head_rows(*ko, *q))
      return none();
    int wcode = 0;
    if (norm) {
      wcode = weight_code(*wq, *q);
      if (wcode < 0 || wk->scalar_type() != wq->scalar_type()) return none();
      for (const Tensor* w : {wq, wk})
        if (w->numel() != kHeadDim || !w->is_contiguous() || w->device() != q->device()) return none();
    }
    for (const Tensor* c : {kc, vc})
      if (c->scalar_type() != q->scalar_type() || c->device() != q->device() || c->dim() != 4 ||
          c->size(2) != k->size(1) || c->size(3) != kHeadDim || !c->is_contiguous())
        return none();
    if (kc->sizes() != vc->sizes() || !slot_list(*slots, *q, tokens)) return none();
    void* const stream = stream_of(*q);
    const int status = unlocked(
        mva_qk_norm_rope_store, ptr(*q), ptr(*qo), q->stride(0), q->stride(1), (int)q->size(1), ptr(*k), ptr(*ko),
        k->stride(0), k->stride(1), ptr(*v), v->stride(0), v->stride(1), (int)k->size(1), (const int64_t*)ptr(*pos),
        (const float*)ptr(*table), table->size(0), kHeadDim, norm ? ptr(*wq) : nullptr, norm ? ptr(*wk) : nullptr,
        wcode, (float)eps, ptr(*kc), ptr(*vc), kc->size(0) * kc->size(1), ptr(*slots),
        slots->scalar_type() == at::kLong, tokens, kHeadDim, code, stream);
    return launched("mva_qk_norm_rope_store", status);
  });
}

// The paged operators' shared tensors, checked as ops._check_paged does.
struct Paged {
  const Tensor *q, *kc, *vc, *bt, *sl, *out;
  int code;
  bool read(PyObject* q_, PyObject* kc_, PyObject* vc_, PyObject* bt_, PyObject* sl_, PyObject* out_) {
    q = plain(q_), kc = plain(kc_), vc = plain(vc_), bt = plain(bt_), sl = plain(sl_), out = plain(out_);
    if (!q || !kc || !vc || !bt || !sl || !out || q->dim() != 3 || out->dim() != 3) return false;
    code = dtype_code(*q);
    if (code < 0) return false;
    for (const Tensor* t : {kc, vc, out})
      if (t->device() != q->device() || t->scalar_type() != q->scalar_type()) return false;
    if (kc->dim() != 4 || vc->sizes() != kc->sizes() || vc->strides() != kc->strides() || kc->stride(3) != 1 ||
        kc->stride(2) != kc->size(3))
      return false;
    return bt->dim() == 2 && bt->stride(1) == 1 && bt->scalar_type() == at::kInt && bt->device() == q->device() &&
           ints(sl);
  }
  bool ints(const Tensor* t) const {
    return t && t->scalar_type() == at::kInt && t->device() == q->device() && t->is_contiguous();
  }
  bool bytes(const Tensor* t) const { return t && t->device() == q->device() && t->is_contiguous(); }
};

int64_t nbytes(const Tensor* t) { return t ? t->numel() * (int64_t)t->element_size() : 0; }
const int32_t* words(const Tensor* t) { return t ? (const int32_t*)ptr(*t) : nullptr; }

// (q, k_cache, v_cache, block_tables, seq_lens, items, num_items, num_waves,
//  merges | None, num_merges, num_part_slots, out, workspace, scale,
//  wave_extra | None, waves_per_group[, key, value, slot_mapping])
PyObject* paged_decode(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Paged p;
    int64_t items_n, waves, merges_n, slots_n, per_group;
    double scale;
    if ((n != 16 && n != 19) || !p.read(a[0], a[1], a[2], a[3], a[4], a[11])) return none();
    const Tensor *items = plain(a[5]), *merges = a[8] == Py_None ? nullptr : plain(a[8]), *ws = plain(a[12]);
    const Tensor* extra = a[14] == Py_None ? nullptr : plain(a[14]);
    if (!p.ints(items) || (a[8] != Py_None && !p.ints(merges)) || (a[14] != Py_None && !p.ints(extra)) || !p.bytes(ws) ||
        !as_int(a[6], &items_n) || !as_int(a[7], &waves) || !as_int(a[9], &merges_n) || !as_int(a[10], &slots_n) ||
        !as_float(a[13], &scale) || !as_int(a[15], &per_group))
      return none();
    const Tensor &q = *p.q, &kc = *p.kc, &out = *p.out;
    void* const stream = stream_of(q);
    int status;
    if (n == 16) {
      status = unlocked(
          mva_paged_decode, ptr(q), q.stride(0), q.stride(1), ptr(kc), ptr(*p.vc), kc.size(0), kc.stride(0),
          kc.stride(1), words(p.bt), p.bt->stride(0), words(p.sl), words(items), items_n, waves, words(extra),
          (int)per_group, words(merges), merges_n, slots_n, ptr(out), out.stride(0), out.stride(1), ptr(*ws),
          nbytes(ws), (int)q.size(1), (int)kc.size(2), (int)q.size(2), (int)kc.size(1), (float)scale, p.code, stream);
    } else {
      const Tensor *k = plain(a[16]), *v = plain(a[17]), *slots = plain(a[18]);
      if (!extra || !k || !v || !slots || k->sizes() != v->sizes() || k->dim() != 3 || k->size(1) != kc.size(2) ||
          k->size(2) != q.size(2) || k->scalar_type() != q.scalar_type() || v->scalar_type() != q.scalar_type() ||
          k->device() != q.device() || v->device() != q.device() || k->stride(2) != 1 || v->stride(2) != 1 ||
          !slot_list(*slots, q, k->size(0)))
        return none();
      status = unlocked(
          mva_paged_decode_store, ptr(q), q.stride(0), q.stride(1), ptr(kc), ptr(*p.vc), kc.size(0), kc.stride(0),
          kc.stride(1), words(p.bt), p.bt->stride(0), words(p.sl), words(items), items_n, waves, words(extra),
          (int)per_group, words(merges), merges_n, slots_n, ptr(out), out.stride(0), out.stride(1), ptr(*ws),
          nbytes(ws), ptr(*k), k->stride(0), k->stride(1), ptr(*v), v->stride(0), v->stride(1), ptr(*slots),
          slots->scalar_type() == at::kLong, k->size(0), (int)q.size(1), (int)kc.size(2), (int)q.size(2),
          (int)kc.size(1), (float)scale, p.code, stream);
    }
    return launched(n == 16 ? "mva_paged_decode" : "mva_paged_decode_store", status);
  });
}

// (q, k_cache, v_cache, block_tables, seq_lens, query_start_loc, num_seqs,
//  max_tiles, workspace, out, scale, planned)
PyObject* paged_prefill(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Paged p;
    int64_t seqs, tiles;
    double scale;
    if (n != 12 || !p.read(a[0], a[1], a[2], a[3], a[4], a[9])) return none();
    const Tensor *qsl = plain(a[5]), *ws = plain(a[8]);
    if (!p.ints(qsl) || !p.bytes(ws) || !as_int(a[6], &seqs) || !as_int(a[7], &tiles) || !as_float(a[10], &scale) ||
        !PyBool_Check(a[11]))
      return none();
    const bool planned = a[11] == Py_True;
    const Tensor &q = *p.q, &kc = *p.kc, &out = *p.out;
    void* const stream = stream_of(q);
    const int status = unlocked(
        planned ? mva_paged_prefill_run : mva_paged_prefill, ptr(q), q.stride(0), q.stride(1), ptr(kc), ptr(*p.vc),
        kc.size(0), kc.stride(0), kc.stride(1), words(p.bt), p.bt->stride(0), words(p.sl), words(qsl), seqs, tiles,
        ptr(*ws), nbytes(ws), ptr(out), out.stride(0), out.stride(1), (int)q.size(1), (int)kc.size(2), (int)q.size(2),
        (int)kc.size(1), (float)scale, p.code, stream);
    return launched(planned ? "mva_paged_prefill_run" : "mva_paged_prefill", status);
  });
}

// (q, k_cache, v_cache, block_tables, seq_lens, query_start_loc, num_seqs,
//  max_tiles, items | None, num_items, num_waves, num_part_slots, out,
//  workspace, scale[, prefill_workgroups, prefill_workspace, planned,
//  wave_extra, merges, num_merges])
PyObject* paged_mixed(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Paged p;
    int64_t seqs, tiles, items_n, waves, slots_n;
    double scale;
    if ((n != 15 && n != 21) || !p.read(a[0], a[1], a[2], a[3], a[4], a[12])) return none();
    const Tensor *qsl = plain(a[5]), *items = a[8] == Py_None ? nullptr : plain(a[8]), *ws = plain(a[13]);
    if (!p.ints(qsl) || (a[8] != Py_None && !p.ints(items)) || !p.bytes(ws) || !as_int(a[6], &seqs) ||
        !as_int(a[7], &tiles) || !as_int(a[9], &items_n) || !as_int(a[10], &waves) || !as_int(a[11], &slots_n) ||
        !as_float(a[14], &scale))
      return none();
    const Tensor &q = *p.q, &kc = *p.kc, &out = *p.out;
    void* const stream = stream_of(q);
    int status;
    if (n == 15) {
      status = unlocked(
          mva_paged_mixed, ptr(q), q.stride(0), q.stride(1), ptr(kc), ptr(*p.vc), kc.size(0), kc.stride(0),
          kc.stride(1), words(p.bt), p.bt->stride(0), words(p.sl), words(qsl), seqs, tiles, words(items), items_n,
          waves, slots_n, ptr(out), out.stride(0), out.stride(1), ptr(*ws), nbytes(ws), (int)q.size(1),
          (int)kc.size(2), (int)q.size(2), (int)kc.size(1), (float)scale, p.code, stream);
    } else {
      const Tensor *pws = plain(a[16]), *extra = plain(a[18]), *merges = plain(a[19]);
      int64_t workgroups, merges_n;
      if (!items || !p.bytes(pws) || !p.ints(extra) || !p.ints(merges) || !as_int(a[15], &workgroups) ||
          !PyBool_Check(a[17]) || !as_int(a[20], &merges_n))
        return none();
      status = unlocked(
          mva_paged_mixed_run, ptr(q), q.stride(0), q.stride(1), ptr(kc), ptr(*p.vc), kc.size(0), kc.stride(0),
          kc.stride(1), words(p.bt), p.bt->stride(0), words(p.sl), words(qsl), seqs, tiles, workgroups, ptr(*pws),
          nbytes(pws), a[17] == Py_True, words(items), items_n, waves, words(extra), words(merges), merges_n, slots_n,
          ptr(out), out.stride(0), out.stride(1), ptr(*ws), nbytes(ws), (int)q.size(1), (int)kc.size(2),
          (int)q.size(2), (int)kc.size(1), (float)scale, p.code, stream);
    }
    return launched(n == 15 ? "mva_paged_mixed" : "mva_paged_mixed_run", status);
  });
}

// (q, k_cache, v_cache, MVA_DTYPE_* of the backend, num_q_heads, num_kv_heads, head_dim, page_size): whether a backend forward's
// query and caches have the layout it takes.
PyObject* forward_inputs_ok(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    int64_t code, hq, hkv, dim, page;
    if (n != 8 || !as_int(a[3], &code) || !as_int(a[4], &hq) || !as_int(a[5], &hkv) || !as_int(a[6], &dim) ||
        !as_int(a[7], &page))
      return none();
    const Tensor *q = plain(a[0]), *kc = plain(a[1]), *vc = plain(a[2]);
    if (!q || !kc || !vc || dtype_code(*q) != code || q->dim() != 3 || q->size(1) != hq || q->size(2) != dim ||
        q->stride(2) != 1)
      return none();
    for (const Tensor* c : {kc, vc})
      if (c->device() != q->device() || c->scalar_type() != q->scalar_type() || c->dim() != 4 || c->size(1) != page ||
          c->size(2) != hkv || c->size(3) != dim || c->stride(3) != 1 || c->stride(2) != dim ||
          c->stride(1) != hkv * dim)
        return none();
    if (kc->sizes() != vc->sizes() || kc->strides() != vc->strides()) return none();
    Py_RETURN_TRUE;
  });
}

// (device index): number of the graph capture that torch's current stream of
// the device is in, or 0.
PyObject* capture_id(PyObject*, PyObject* const* a, Py_ssize_t n) {
  int64_t device;
  if (n != 1 || !as_int(a[0], &device)) return PyErr_Format(PyExc_TypeError, "capture_id takes a device index");
  unsigned long long id = 0;
  try {
    hipStreamCaptureStatus status;
    const hipStream_t stream = c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream();
    if (hipStreamGetCaptureInfo(stream, &status, &id) != hipSuccess || status != hipStreamCaptureStatusActive) id = 0;
  } catch (const std::exception& error) {
    return PyErr_Format(PyExc_RuntimeError, "%s", error.what());
  }
  return PyLong_FromUnsignedLongLong(id);
}

#define MVA_METHOD(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {MVA_METHOD(silu_and_mul),       MVA_METHOD(rms_norm),      MVA_METHOD(fused_add_rms_norm),
                          MVA_METHOD(qk_norm_rope_store), MVA_METHOD(paged_decode),  MVA_METHOD(paged_prefill),
                          MVA_METHOD(paged_mixed),        MVA_METHOD(forward_inputs_ok), MVA_METHOD(capture_id),
                          {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "mva_host", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_mva_host(void) {
  PyObject* m = PyModule_Create(&kModule);
  if (m != nullptr && PyModule_AddIntConstant(m, "ABI_VERSION", MVA_HOST_ABI_VERSION) != 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
