// front.cpp — the caller's side of the mixers' operators (attention over paged rows and latents, recurrences, mixture of experts) as a
// Python module: operands checked, results and workspaces allocated, the argument block filled in and the library called without
// the interpreter in between.  The operators' Python functions (_C/kernel) call it first: what they return for operands that pass every
// check comes from here, everything else (None is returned) goes on in Python, which says what it refuses and why.  A check here is the
// Python function's own, so that nothing is taken here that would be refused there.
// Host time bounds short calls.  Caller's time of a call, us, in Python and from here (the library's launch is 3 of it, or 5 where there are two):
// state_scan of single tokens 14.9 and 6.3 (its kernel 5), latent and paged attention 14.0 and 6.1, with key splits 18.0 and 9.6, a
// gated recurrence's step 18.2 and 9.8, the five calls of a mixture of experts 53 and 32.
// No state but the library's addresses: threads and streams call it as they call the library, which runs without the interpreter's lock.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <ATen/ops/empty.h>
#include <c10/hip/HIPFunctions.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/hydra_hip.h"
#include "../../include/hydra_mix.h"

namespace {

#define HX_ENTRIES(X)                                                                                                            \
  X(hxm_latent_attention) X(hxm_latent_attention_plan) X(hxm_biased_attention) X(hxm_biased_attention_plan) X(hxm_state_scan)      \
  X(hxm_state_scan_workspace) X(hxm_gated_recurrence) X(hxm_gated_recurrence_batch_workspace) X(hxm_router_topk) X(hxm_moe_plan) \
  X(hxm_grouped_linear) X(hxm_moe_combine)
struct Entries {
#define X(name) decltype(&::name) name = nullptr;
  HX_ENTRIES(X)
#undef X
} lib;
PyObject* check = nullptr;                 // _lib.mix_check(status, what): raises

// What a call's operands are read with; `ok` falls where Python has to decide.
struct Args {
  PyObject* const* v;
  int device = -1;                         // the thread's current one, asked for when a device tensor is there: the runtime is up then
  bool ok = true;

  explicit Args(PyObject* const* args) : v(args) {}
  const at::Tensor* tensor(PyObject* o) {
    if (!THPVariable_Check(o)) { ok = false; return nullptr; }
    const at::Tensor& t = THPVariable_Unpack(o);
    // (tensors that are not plain memory of the current device: functional transforms, subclasses that dispatch to Python, other layouts)
    constexpr c10::DispatchKeySet strange({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                           c10::DispatchKey::Batched, c10::DispatchKey::Functionalize, c10::DispatchKey::Negative, c10::DispatchKey::Conjugate});
    if (!t.defined() || !t.is_cuda() || t.layout() != c10::kStrided || t.key_set().has_any(strange)) { ok = false; return &t; }
    if (device < 0) device = c10::hip::current_device();
    if (t.get_device() != device) ok = false;
    return &t;
  }
  const at::Tensor* tensor(int i) { return tensor(v[i]); }
  const at::Tensor* maybe(int i) { return v[i] == Py_None ? nullptr : tensor(v[i]); }
  int64_t integer(int i, int64_t lo = INT32_MIN, int64_t hi = INT32_MAX) {
    if (!PyLong_CheckExact(v[i])) { ok = false; return 0; }
    int overflow = 0;
    const int64_t n = PyLong_AsLongLongAndOverflow(v[i], &overflow);
    if (overflow || n < lo || n > hi) ok = false;
    return n;
  }
  int64_t integer_or_none(int i) { return v[i] == Py_None ? 0 : integer(i); }
  float number(int i) {
    if (PyFloat_CheckExact(v[i])) return (float)PyFloat_AS_DOUBLE(v[i]);
    return (float)integer(i);
  }
  bool is(int i, const char* name) { return PyUnicode_Check(v[i]) && PyUnicode_CompareWithASCIIString(v[i], name) == 0; }
  // a text's place among `names`
  template <size_t N>
  int one_of(int i, const char* const (&names)[N]) {
    for (size_t k = 0; k < N; ++k)
      if (is(i, names[k])) return (int)k;
    ok = false;
    return 0;
  }
  void need(bool holds) { ok = ok && holds; }
  const int32_t* ints(const at::Tensor* t, int64_t n) {
    if (!ok) return nullptr;
    need(t->scalar_type() == at::kInt && t->is_contiguous() && t->numel() == n);
    return (const int32_t*)t->data_ptr();
  }
  const float* floats(const at::Tensor* t, int64_t n) {
    if (!ok || !t) return nullptr;
    need(t->scalar_type() == at::kFloat && t->is_contiguous() && t->numel() == n);
    return (const float*)t->data_ptr();
  }
  // [n, width] with contiguous rows
  void rows(const at::Tensor* t, int64_t n, int64_t width) { need(ok && t->dim() == 2 && t->size(0) == n && t->size(1) == width && t->stride(1) == 1); }
  int act(const at::Tensor* t) {           // activations are float32 or bfloat16
    if (!ok) return 0;
    const auto type = t->scalar_type();
    need(type == at::kFloat || type == at::kBFloat16);
    return type == at::kFloat ? HX_F32 : HX_BF16;
  }
  at::Tensor empty(at::IntArrayRef shape, at::ScalarType type) {
    return at::empty(shape, at::TensorOptions().dtype(type).device(c10::Device(c10::kCUDA, (c10::DeviceIndex)device)));
  }
  void* stream() const { return (void*)c10::hip::getCurrentHIPStreamMasqueradingAsCUDA((c10::DeviceIndex)device).stream(); }
};

PyObject* declined() { Py_RETURN_NONE; }
PyObject* failed(int status, const char* what) {
  PyObject* r = PyObject_CallFunction(check, "is", status, what);
  if (r) {                                 // (it raises for every status that is not 0)
    Py_DECREF(r);
    PyErr_SetString(PyExc_RuntimeError, what);
  }
  return nullptr;
}
template <typename F>
int without_lock(F call) {
  PyThreadState* saved = PyEval_SaveThread();
  const int status = call();
  PyEval_RestoreThread(saved);
  return status;
}
const void* at_or_null(const at::Tensor* t) { return t ? t->data_ptr() : nullptr; }

// The batch's state (stream_ops.SequenceState)
struct Sequences {
  PyObject *state = nullptr, *slots = nullptr, *tok_seq = nullptr;
  explicit Sequences(PyObject* o) {
    state = PyObject_GetAttrString(o, "state");
    slots = PyObject_GetAttrString(o, "slots");
    tok_seq = PyObject_GetAttrString(o, "tok_seq");
    if (!state || !slots || !tok_seq) PyErr_Clear();
  }
  bool all() const { return state && slots && tok_seq; }
  ~Sequences() {
    Py_XDECREF(state);
    Py_XDECREF(slots);
    Py_XDECREF(tok_seq);
  }
};

// (q, cache, tok_seq, positions, q_cu, block_table, cu_block_lens, scale, window, max_q_len, gate_pre, out, max_kv_len, sinks)
PyObject* latent_attention(PyObject*, PyObject* const* v, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  if (n_args != 14) return declined();
  Args x(v);
  const at::Tensor *q = x.tensor(0), *cache = x.tensor(1), *tok_seq = x.tensor(2), *positions = x.tensor(3), *q_cu = x.tensor(4), *table = x.tensor(5),
                   *cu_blocks = x.tensor(6), *gate = x.maybe(10), *given = x.maybe(11), *sinks = x.maybe(13);
  hxm_latent_attn_args a{};
  a.scale = x.number(7);
  a.window = (int32_t)x.integer_or_none(8);
  a.max_q_len = (int32_t)x.integer(9);
  a.max_kv_len = (int32_t)x.integer(12);
  if (!x.ok) return declined();
  x.need(q->dim() == 3 && q->stride(2) == 1 && cache->scalar_type() == q->scalar_type());
  if (!x.ok) return declined();
  const int64_t T = q->size(0), H = q->size(1), R = q->size(2), n_seq = q_cu->numel() - 1;
  x.need(R <= HXM_MAX_LATENT && T <= INT32_MAX && H <= INT32_MAX && n_seq <= INT32_MAX);
  a.tok_seq = x.ints(tok_seq, T);
  a.positions = x.ints(positions, T);
  a.q_cu = x.ints(q_cu, n_seq + 1);
  a.cu_block_lens = x.ints(cu_blocks, n_seq + 1);
  a.block_table = x.ints(table, table->numel());
  a.sinks = x.floats(sinks, H);
  if (given) x.need(given->sizes() == q->sizes() && given->scalar_type() == q->scalar_type() && given->stride(2) == 1);
  if (gate) {
    x.need(gate->scalar_type() == q->scalar_type() && gate->dim() == 2 && gate->size(0) == T && gate->size(1) >= H && gate->stride(1) == 1);
    if (!x.ok) return declined();
    a.gate_pre = gate->data_ptr();
    a.gate_stride = gate->stride(0);
  }
  x.need(cache->dim() == 4 && cache->size(2) == 1 && cache->size(3) >= R && cache->stride(3) == 1 && cache->size(1) <= INT32_MAX);
  a.dtype = x.act(q);
  if (!x.ok) return declined();
  const at::Tensor out = given ? *given : x.empty({T, H, R}, q->scalar_type());
  a.out = out.data_ptr();
  a.q = q->data_ptr();
  a.cache = cache->data_ptr();
  a.q_token_stride = q->stride(0);
  a.q_head_stride = q->stride(1);
  a.out_token_stride = out.stride(0);
  a.out_head_stride = out.stride(1);
  a.cache_block_stride = cache->stride(0);
  a.cache_row_stride = cache->stride(1);
  a.block_size = (int32_t)cache->size(1);
  a.n_tokens = (int32_t)T;
  a.n_seq = (int32_t)n_seq;
  a.n_heads = (int32_t)H;
  a.kv_rank = (int32_t)R;
  a.n_splits = 1;
  at::Tensor ws;
  if (a.max_kv_len > 0) {                  // (0: unknown, no key splits)
    int32_t splits = 1;
    int64_t need = 0;
    if (const int rc = lib.hxm_latent_attention_plan(&a, &splits, &need)) return failed(rc, "latent_attention_plan");
    if (splits > 1) {
      ws = x.empty({need}, at::kFloat);
      const int64_t wide = (R + 15) / 16 * 16;
      a.n_splits = splits;
      a.ws_o = (float*)ws.data_ptr();
      a.ws_ml = a.ws_o + need / (wide + 2) * wide;
    }
  }
  void* stream = x.stream();
  if (const int rc = without_lock([&] { return lib.hxm_latent_attention(&a, stream); })) return failed(rc, "latent_attention");
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// (q, key_cache, value_cache, vdim, tok_seq, positions, q_cu, block_table, cu_block_lens, scale, slopes, mask, mask_size, max_q_len, kv_heads,
//  max_kv_len, form, softcap, head_scale, sinks)
PyObject* biased_attention(PyObject*, PyObject* const* v, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  if (n_args != 20) return declined();
  Args x(v);
  const at::Tensor *q = x.tensor(0), *keys = x.tensor(1), *values = x.tensor(2), *tok_seq = x.tensor(4), *positions = x.tensor(5), *q_cu = x.tensor(6),
                   *table = x.tensor(7), *cu_blocks = x.tensor(8), *slopes = x.maybe(10), *head_scale = x.maybe(18), *sinks = x.maybe(19);
  hxm_biased_attn_args a{};
  static const char* const kMasks[] = {"causal", "window", "chunk"};
  static const char* const kForms[] = {"auto", "rows", "tile"};
  const int64_t vdim = x.integer(3);
  a.scale = x.number(9);
  a.mask_kind = x.one_of(11, kMasks);
  a.mask_size = (int32_t)x.integer(12);
  a.max_q_len = (int32_t)x.integer(13);
  int64_t G = x.integer_or_none(14);
  const int32_t max_kv_len = (int32_t)x.integer(15);
  a.form = x.one_of(16, kForms);
  a.softcap = x.number(17);
  if (!x.ok) return declined();
  x.need(q->dim() == 3 && q->is_contiguous() && keys->scalar_type() == q->scalar_type() && values->scalar_type() == q->scalar_type() && keys->dim() == 4);
  if (!x.ok) return declined();
  const int64_t T = q->size(0), H = q->size(1), D = q->size(2), n_seq = q_cu->numel() - 1;
  if (!G) G = keys->size(2);
  x.need(values->strides() == keys->strides() && G > 0 && H % G == 0 && keys->size(2) >= G && keys->stride(3) == 1 && keys->stride(1) != 0);
  if (!x.ok) return declined();
  x.need(keys->stride(0) % keys->stride(1) == 0 && keys->stride(0) / keys->stride(1) == keys->size(1));
  x.need(D <= keys->size(3) && vdim <= keys->size(3) && vdim > 0 && T <= INT32_MAX && H <= INT32_MAX && n_seq <= INT32_MAX && keys->size(1) <= INT32_MAX);
  x.need(a.mask_kind == 0 || a.mask_size >= 1);
  a.tok_seq = x.ints(tok_seq, T);
  a.positions = x.ints(positions, T);
  a.q_cu = x.ints(q_cu, n_seq + 1);
  a.cu_block_lens = x.ints(cu_blocks, n_seq + 1);
  a.block_table = x.ints(table, table->numel());
  a.slopes = x.floats(slopes, H);
  a.head_scale = x.floats(head_scale, H);
  a.sinks = x.floats(sinks, H);
  a.dtype = x.act(q);
  if (!x.ok) return declined();
  const at::Tensor out = x.empty({T, H, vdim}, q->scalar_type());
  a.out = out.data_ptr();
  a.q = q->data_ptr();
  a.key_cache = keys->data_ptr();
  a.value_cache = values->data_ptr();
  a.cache_block_stride = keys->stride(0);
  a.cache_row_stride = keys->stride(1);
  a.head_stride = keys->stride(2);
  a.block_size = (int32_t)keys->size(1);
  a.n_tokens = (int32_t)T;
  a.n_heads = (int32_t)H;
  a.kv_heads = (int32_t)G;
  a.dim = (int32_t)D;
  a.vdim = (int32_t)vdim;
  a.n_seq = (int32_t)n_seq;
  a.n_splits = 1;
  at::Tensor ws;
  int32_t splits = 1;
  int64_t need = 0;
  if (const int rc = lib.hxm_biased_attention_plan(&a, max_kv_len, &splits, &need)) return failed(rc, "biased_attention_plan");
  if (splits > 1) {
    ws = x.empty({need}, at::kFloat);
    const int64_t wide = (vdim + 15) / 16 * 16;
    a.n_splits = splits;
    a.ws_o = (float*)ws.data_ptr();
    a.ws_ml = a.ws_o + need / (wide + 2) * wide;
  }
  void* stream = x.stream();
  if (const int rc = without_lock([&] { return lib.hxm_biased_attention(&a, stream); })) return failed(rc, "biased_attention");
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// (mode, q, k, v, decay, seq, offset, q_cu, positions, heads, qk_heads, dim, vdim, vscale, beta, bonus)
PyObject* state_scan(PyObject*, PyObject* const* v, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  if (n_args != 16) return declined();
  Args x(v);
  const Sequences seq(v[5]);
  if (!seq.all()) return declined();
  const at::Tensor *q = x.tensor(1), *k = x.tensor(2), *val = x.tensor(3), *decay = x.tensor(4), *state = x.tensor(seq.state), *slots = x.tensor(seq.slots),
                   *tok_seq = x.tensor(seq.tok_seq), *q_cu = x.tensor(7), *positions = x.tensor(8), *vscale = x.maybe(13), *beta = x.maybe(14), *bonus = x.maybe(15);
  hxm_state_scan_args a{};
  static const char* const kModes[] = {"decay", "bonus", "delta"};
  a.mode = x.one_of(0, kModes);
  const int64_t offset = x.integer(6, 0, INT64_MAX);
  const int64_t heads = x.integer(9, 1), qk_heads = x.integer(10, 1), dim = x.integer(11, 1), vdim = x.integer(12, 1);
  if (!x.ok || heads * dim > INT32_MAX || heads * vdim > INT32_MAX) return declined();
  x.need((a.mode != 2 || beta) && (a.mode != 1 || bonus) && q->dim() == 2);
  if (!x.ok) return declined();
  const int64_t T = q->size(0), n_seq = q_cu->numel() - 1;
  x.rows(q, T, qk_heads * dim);
  x.rows(k, T, qk_heads * dim);
  x.rows(val, T, heads * vdim);
  a.decay_per_channel = decay->dim() == 2 && decay->size(1) == heads * dim && dim > 1;
  a.decay = x.floats(decay, T * heads * (a.decay_per_channel ? dim : 1));
  a.vscale = x.floats(vscale, T * heads);
  a.beta = x.floats(beta, T * heads);
  a.bonus = x.floats(bonus, heads * dim);
  a.q_cu = x.ints(q_cu, n_seq + 1);
  a.positions = x.ints(positions, T);
  a.slots = x.ints(slots, n_seq);
  x.ints(tok_seq, T);
  x.need(state->scalar_type() == at::kFloat && state->dim() == 3 && state->is_contiguous() && n_seq <= INT32_MAX);
  if (!x.ok) return declined();
  const int64_t piece = heads * dim * vdim, slot = state->size(1) * state->size(2);
  x.need(heads * dim <= INT64_MAX / 4 / vdim && offset <= slot && piece <= slot - offset);
  a.q_dtype = x.act(q);
  a.k_dtype = x.act(k);
  a.v_dtype = x.act(val);
  if (!x.ok) return declined();
  const at::Tensor out = x.empty({T, heads * vdim}, at::kFloat);
  a.out = (float*)out.data_ptr();
  a.q = q->data_ptr();
  a.k = k->data_ptr();
  a.v = val->data_ptr();
  a.q_stride = q->stride(0);
  a.k_stride = k->stride(0);
  a.v_stride = val->stride(0);
  a.state = (float*)state->data_ptr() + offset;
  a.slot_stride = state->stride(0);
  a.n_tokens = T;
  a.n_seq = (int32_t)n_seq;
  a.heads = (int32_t)heads;
  a.qk_heads = (int32_t)qk_heads;
  a.dim = (int32_t)dim;
  a.vdim = (int32_t)vdim;
  at::Tensor ws;
  if (T > n_seq) {                         // portions of prompts: what their chunks need is made in a launch ahead
    a.ws_floats = lib.hxm_state_scan_workspace(&a);
    if (a.ws_floats > 0) {
      ws = x.empty({a.ws_floats}, at::kFloat);
      a.ws = (float*)ws.data_ptr();
    }
  }
  void* stream = x.stream();
  if (const int rc = without_lock([&] { return lib.hxm_state_scan(&a, stream); })) return failed(rc, "state_scan");
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// (q_pre, f_pre, v, f_bias, low, norm_w, eps, seq, state_row, q_cu, positions, heads, dim, vdim, max_q_len)
PyObject* gated_recurrence(PyObject*, PyObject* const* v, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  if (n_args != 15) return declined();
  Args x(v);
  const Sequences seq(v[7]);
  if (!seq.all()) return declined();
  const at::Tensor *q = x.tensor(0), *f = x.tensor(1), *val = x.tensor(2), *f_bias = x.tensor(3), *low = x.tensor(4), *norm_w = x.tensor(5),
                   *state = x.tensor(seq.state), *slots = x.tensor(seq.slots), *q_cu = x.tensor(9), *positions = x.tensor(10);
  const float eps = x.number(6);
  const int64_t row = x.integer(8, 0), heads = x.integer(11, 1), dim = x.integer(12, 1), vdim = x.integer(13, 1), longest = x.integer(14);
  if (!x.ok || heads * dim > INT32_MAX || heads * vdim > INT32_MAX || q->dim() != 2) return declined();
  const int64_t T = q->size(0), n_seq = q_cu->numel() - 1;
  const int dtype = x.act(q);
  x.rows(q, T, heads * dim);
  x.rows(f, T, heads * dim);
  x.rows(val, T, heads * vdim);
  x.need(f->scalar_type() == q->scalar_type() && val->scalar_type() == q->scalar_type() && n_seq <= INT32_MAX);
  const float *bias_at = x.floats(f_bias, heads * dim), *low_at = x.floats(low, heads * dim), *norm_at = x.floats(norm_w, vdim);
  const int32_t *cu_at = x.ints(q_cu, n_seq + 1), *pos_at = x.ints(positions, T), *slots_at = x.ints(slots, n_seq);
  x.need(state->scalar_type() == at::kFloat && state->dim() == 3 && state->is_contiguous() && heads * dim <= INT64_MAX / 4 / vdim);
  if (!x.ok) return declined();
  x.need(state->size(2) >= heads * dim * vdim && row < state->size(1));
  if (!x.ok) return declined();
  const at::Tensor out = x.empty({T, heads * vdim}, q->scalar_type());
  float* base = (float*)state->data_ptr() + row * state->stride(1);
  // partial results of the key channels' parts, or results and what chunks need
  const int64_t floats = lib.hxm_gated_recurrence_batch_workspace((int32_t)n_seq, T, (int32_t)heads, (int32_t)dim, (int32_t)vdim, (int32_t)longest, dtype);
  const at::Tensor ws = x.empty({std::max<int64_t>(floats, 1)}, at::kFloat);
  void* stream = x.stream();
  const int rc = without_lock([&] {
    return lib.hxm_gated_recurrence(out.data_ptr(), q->data_ptr(), q->stride(0), f->data_ptr(), f->stride(0), val->data_ptr(), val->stride(0), bias_at, low_at,
                                    norm_at, eps, base, state->stride(0), cu_at, pos_at, slots_at, (int32_t)n_seq, T, (int32_t)heads, (int32_t)dim,
                                    (int32_t)vdim, (int32_t)longest, (float*)ws.data_ptr(), floats, dtype, stream);
  });
  if (rc) return failed(rc, "gated_recurrence");
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

PyObject* wrapped(std::initializer_list<at::Tensor> many) {
  PyObject* r = PyTuple_New((Py_ssize_t)many.size());
  Py_ssize_t i = 0;
  for (const at::Tensor& t : many) {
    PyObject* o = r ? THPVariable_Wrap(t) : nullptr;
    if (!o) {
      Py_XDECREF(r);
      return nullptr;
    }
    PyTuple_SET_ITEM(r, i++, o);
  }
  return r;
}

// (x, w, bias, top)
PyObject* router_topk(PyObject*, PyObject* const* v, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  if (n_args != 4) return declined();
  Args x(v);
  const at::Tensor *h = x.tensor(0), *w = x.tensor(1), *bias = x.maybe(2);
  const int64_t top = x.integer(3, 0);
  if (!x.ok || w->dim() != 2) return declined();
  const int64_t E = w->size(0), K = w->size(1);
  x.need(h->scalar_type() == at::kFloat && h->dim() == 2 && E <= INT32_MAX);
  if (!x.ok) return declined();
  const int64_t T = h->size(0);
  x.rows(h, T, K);
  const float *w_at = x.floats(w, E * K), *bias_at = x.floats(bias, E);
  if (!x.ok) return declined();
  const at::Tensor weights = x.empty({T, top}, at::kFloat), experts = x.empty({T, top}, at::kInt);
  void* stream = x.stream();
  const int rc = without_lock([&] {
    return lib.hxm_router_topk((const float*)h->data_ptr(), h->stride(0), w_at, bias_at, T, K, (int32_t)E, (int32_t)top, (float*)weights.data_ptr(),
                               (int32_t*)experts.data_ptr(), stream);
  });
  if (rc) return failed(rc, "router_topk");
  return wrapped({weights, experts});
  END_HANDLE_TH_ERRORS
}

// (experts, n_experts)
PyObject* moe_plan(PyObject*, PyObject* const* v, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  if (n_args != 2) return declined();
  Args x(v);
  const at::Tensor* experts = x.tensor(0);
  const int64_t E = x.integer(1, 0, INT32_MAX - 1);
  if (!x.ok) return declined();
  x.need(experts->dim() == 2);
  const int32_t* at = x.ints(experts, experts->numel());
  if (!x.ok) return declined();
  const int64_t T = experts->size(0), top = experts->size(1);
  const at::Tensor seg = x.empty({E + 1}, at::kInt), row_of = x.empty({T, top}, at::kInt), src = x.empty({T * top}, at::kInt);
  void* stream = x.stream();
  const int rc = without_lock([&] {
    return lib.hxm_moe_plan(at, T, (int32_t)top, (int32_t)E, (int32_t*)seg.data_ptr(), (int32_t*)row_of.data_ptr(), (int32_t*)src.data_ptr(), stream);
  });
  if (rc) return failed(rc, "moe_plan");
  return wrapped({seg, row_of, src});
  END_HANDLE_TH_ERRORS
}

// (x, w, seg, max_rows, src, act, limit, alpha, up_shift)
PyObject* grouped_linear(PyObject*, PyObject* const* v, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  if (n_args != 9) return declined();
  Args x(v);
  const at::Tensor *in = x.tensor(0), *w = x.tensor(1), *seg = x.tensor(2), *src = x.maybe(4);
  const int64_t rows = x.integer(3, 0);
  static const char* const kActs[] = {"none", "relu2", "glu"};
  const int act = x.one_of(5, kActs);
  const float limit = x.number(6), alpha = x.number(7), up_shift = x.number(8);
  if (!x.ok) return declined();
  x.need(in->dim() == 2 && in->stride(1) == 1 && w->dim() == 3 && w->is_contiguous() && w->scalar_type() == in->scalar_type());
  if (!x.ok) return declined();
  const int64_t E = w->size(0), N = w->size(1), K = w->size(2);
  x.need(K == in->size(1) && E < INT32_MAX && (src || in->size(0) >= rows) && (act != 2 || N % 32 == 0));
  const int32_t *seg_at = x.ints(seg, E + 1), *src_at = nullptr;
  if (src) {
    src_at = x.ints(src, src->numel());
    x.need(src->numel() >= rows);
  }
  const int dtype = x.act(in);
  if (!x.ok) return declined();
  const at::Tensor y = x.empty({rows, act == 2 ? N / 2 : N}, in->scalar_type());
  void* stream = x.stream();
  const int rc = without_lock([&] {
    return lib.hxm_grouped_linear(y.data_ptr(), in->data_ptr(), in->stride(0), src_at, w->data_ptr(), seg_at, rows, (int32_t)E, N, K, act, limit, alpha, up_shift,
                                  dtype, stream);
  });
  if (rc) return failed(rc, "grouped_linear");
  return THPVariable_Wrap(y);
  END_HANDLE_TH_ERRORS
}

// (y, row_of, weights, shared, shared_gate, identity)
PyObject* moe_combine(PyObject*, PyObject* const* v, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  if (n_args != 6) return declined();
  Args x(v);
  const at::Tensor *y = x.tensor(0), *row_of = x.tensor(1), *weights = x.tensor(2), *shared = x.maybe(3), *gate = x.maybe(4), *identity = x.maybe(5);
  if (!x.ok) return declined();
  x.need(y->dim() == 2 && y->is_contiguous() && row_of->dim() == 2 && weights->sizes() == row_of->sizes());
  const int32_t* row_at = x.ints(row_of, row_of->numel());
  const float* weights_at = x.floats(weights, row_of->numel());
  if (!x.ok) return declined();
  const int64_t T = row_of->size(0), top = row_of->size(1), W = y->size(1);
  if (!shared) gate = nullptr;
  if (shared) x.need(shared->dim() == 2 && shared->size(0) == T && shared->size(1) == W && shared->scalar_type() == y->scalar_type() && shared->is_contiguous());
  if (gate) x.need(gate->scalar_type() == at::kFloat && gate->dim() >= 1 && gate->size(0) == T);
  if (identity) x.need(identity->scalar_type() == y->scalar_type() && identity->dim() == 2 && identity->size(0) == T && identity->size(1) >= W && identity->stride(1) == 1);
  const int dtype = x.act(y);
  if (!x.ok) return declined();
  const at::Tensor out = x.empty({T, W}, y->scalar_type());
  void* stream = x.stream();
  const int rc = without_lock([&] {
    return lib.hxm_moe_combine(out.data_ptr(), y->data_ptr(), row_at, weights_at, at_or_null(shared), (const float*)at_or_null(gate), gate ? gate->stride(0) : 0,
                               at_or_null(identity), identity ? identity->stride(0) : 0, T, (int32_t)top, W, dtype, stream);
  });
  if (rc) return failed(rc, "moe_combine");
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// ({name: address}, mix_check): the entry points of the library that the binding has opened
PyObject* bind(PyObject*, PyObject* const* v, Py_ssize_t n_args) {
  if (n_args != 2 || !PyDict_Check(v[0])) {
    PyErr_SetString(PyExc_TypeError, "bind(addresses, check)");
    return nullptr;
  }
#define X(name)                                                                                                \
  {                                                                                                            \
    PyObject* o = PyDict_GetItemString(v[0], #name);                                                           \
    if (!o) return PyErr_Format(PyExc_KeyError, "%s", #name);                                                  \
    lib.name = reinterpret_cast<decltype(lib.name)>(PyLong_AsVoidPtr(o));                                      \
  }
  HX_ENTRIES(X)
#undef X
  if (PyErr_Occurred()) return nullptr;
  Py_INCREF(v[1]);
  Py_XDECREF(check);
  check = v[1];
  Py_RETURN_NONE;
}

#define X(name) #name,
const char* const kEntries[] = {HX_ENTRIES(X)};
#undef X

#define METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {METHOD(bind), METHOD(latent_attention), METHOD(biased_attention), METHOD(state_scan), METHOD(gated_recurrence), METHOD(router_topk),
                         METHOD(moe_plan), METHOD(grouped_linear), METHOD(moe_combine), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_hydra_front", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// What this was compiled for: the binding asks before it takes this for a module.
#define TEXT(x) #x
#define TEXT_OF(x) TEXT(x)
extern "C" __attribute__((visibility("default"))) const char* hydra_front_built_for() {
  return "ABI " TEXT_OF(HXM_ABI_VERSION) ", torch " HYDRA_TORCH_VERSION ", Python " TEXT_OF(PY_MAJOR_VERSION) "." TEXT_OF(PY_MINOR_VERSION);
}

PyMODINIT_FUNC PyInit__hydra_front() {
  PyObject* m = PyModule_Create(&module);
  if (!m) return nullptr;
  PyObject* names = PyTuple_New((Py_ssize_t)std::size(kEntries));
  for (size_t i = 0; names && i < std::size(kEntries); ++i) PyTuple_SET_ITEM(names, (Py_ssize_t)i, PyUnicode_FromString(kEntries[i]));
  if (!names || PyModule_AddObject(m, "entries", names) < 0) return nullptr;
  return m;
}
