// The operators that small steps consist of, called without a Python frame per argument: the checks of the functions of the
// same names in _C.py / _C_mixers.py, their scratch allocation and the library call, in C++.
//
// Why: a launch costs the host 3 us; a call through the Python functions cost 7 to 11 us, of which ctypes takes 1 and the
// checks, data pointers and the device guard the rest, so that a decode step of two conversations waited for the host (21 us
// a layer, 12.6 on the GPU).  Measured, us a pass of calls, before / now: cache write + attention of a decode step 20.9 /
// 16.6, of a prompt of 40 tokens 21.0 / 15.7; the delta rule with its convolution and norm 34.9 / 23.4; experts 27.4 / 21.9;
// gated linear attention 28.7 / 21.3; the mixers' attention 15.3 / 8.3.  (Cache write and attention are one call where their launches
// are: prefill_attention_and_cache, paged_attention_and_cache.)
//
// A function takes a call only if every argument is of the plain kind (exact tensors on the current device, Python numbers)
// and passes every check; otherwise it returns None before anything happened and the Python function goes on, which knows
// the other forms and words the refusals.  It returns the library's status otherwise.  Leaving a call is a throw, 2 us: common forms that
// it does not take (slopes, sigmoid weights, values inside the key rows) are not offered to it.
#include <Python.h>

#include <ATen/ATen.h>
#include <hip/hip_runtime_api.h>
#include <torch/csrc/autograd/python_variable.h>

#include "splitwise_hip.h"
#include "splitwise_mixers.h"

namespace {

#define STEP_OPS(X)                                                                                                     \
  X(sw_reshape_and_cache) X(sw_paged_attention_v1) X(sw_prefill_attention) X(sw_prefill_attention_and_cache) X(sw_paged_attention_and_cache) X(swm_causal_conv) X(swm_gated_delta)        \
  X(swm_gated_delta_chunked) X(swm_gated_delta_chunked_workspace_floats) X(swm_head_norm_gate_act) X(swm_group_pairs)   \
  X(swm_expert_up_weighted) X(swm_expert_down_weighted) X(swm_masked_attention) X(swm_sink_attention)                   \
  X(swm_masked_attention_workspace_floats) X(swm_gla) X(swm_gla_workspace_floats) X(swm_lightning) X(swm_retention)     \
  X(swm_lightning_workspace_floats)
// entry points of the libraries, set by bind() when one is loaded
#define DECLARE(name) decltype(&::name) name##_at = nullptr;
STEP_OPS(DECLARE)
#undef DECLARE

PyObject* g_raw_stream = nullptr;                  // torch._C._cuda_getCurrentRawStream
PyObject *s_q_start, *s_ctx_len, *s_token_seq, *s_state_slot, *s_block_tables, *s_max_state_slot, *s_max_query_len,
    *s_max_pages_used, *s_max_page_id;

using at::Tensor;
struct NotTaken {};                                // thrown where a call is left to the Python function
inline void take(bool ok) {
  if (!ok) throw NotTaken{};
}

// The arguments of one call.
struct Args {
  PyObject* const* a;
  int device = -1;
  Args(PyObject* const* args, Py_ssize_t n, Py_ssize_t want) : a(args) {
    take(n == want && hipGetDevice(&device) == hipSuccess);
  }
  const Tensor& own(PyObject* o) const {
    take(THPVariable_CheckExact(o));
    const Tensor& t = THPVariable_Unpack(o);
    take(t.is_cuda() && t.get_device() == device && t.layout() == at::kStrided);
    return t;
  }
  const Tensor& tensor(int i) const { return own(a[i]); }
  const Tensor* optional(int i) const { return a[i] == Py_None ? nullptr : &own(a[i]); }
  static int64_t integer(PyObject* o) {
    take(PyLong_Check(o));
    const long long v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) {
      PyErr_Clear();
      throw NotTaken{};
    }
    return v;
  }
  int i32(int i) const {
    const int64_t v = integer(a[i]);
    take(v >= INT32_MIN && v <= INT32_MAX);
    return (int)v;
  }
  static float real(PyObject* o) {
    take(PyFloat_Check(o) || PyLong_CheckExact(o));
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) {
      PyErr_Clear();
      throw NotTaken{};
    }
    return (float)v;
  }
  float f32(int i) const { return real(a[i]); }
  bool flag(int i) const {
    take(PyBool_Check(a[i]));
    return a[i] == Py_True;
  }
  void* stream() const {
    PyObject* index = PyLong_FromLong(device);
    PyObject* handle = index ? PyObject_CallOneArg(g_raw_stream, index) : nullptr;
    Py_XDECREF(index);
    void* p = handle ? PyLong_AsVoidPtr(handle) : nullptr;
    Py_XDECREF(handle);
    if (PyErr_Occurred()) {
      PyErr_Clear();
      throw NotTaken{};
    }
    return p;
  }
};

// The step's layout: what _ragged_ok checks.
struct Ragged {
  PyObject* held[5] = {};
  const Tensor *q_start, *ctx_len, *token_seq, *state_slot, *block_tables = nullptr;
  PyObject* batch;
  const Args& args;
  int n;
  Ragged(const Args& c, PyObject* b, int64_t rows) : batch(b), args(c) {
    try {
      q_start = part(0, s_q_start);
      ctx_len = part(1, s_ctx_len);
      token_seq = part(2, s_token_seq);
      state_slot = part(3, s_state_slot);
      const int64_t seqs = ctx_len->numel();
      take(q_start->numel() == seqs + 1 && token_seq->numel() == rows && state_slot->numel() == seqs && seqs <= INT32_MAX);
      n = (int)seqs;
    } catch (...) {
      release();
      throw;
    }
  }
  Ragged(const Ragged&) = delete;
  ~Ragged() { release(); }
  void release() {
    for (PyObject*& h : held) Py_CLEAR(h);
  }
  PyObject* get(PyObject* name) const {
    PyObject* o = PyObject_GetAttr(batch, name);
    if (o == nullptr) {
      PyErr_Clear();
      throw NotTaken{};
    }
    return o;
  }
  const Tensor* part(int i, PyObject* name) {
    held[i] = get(name);
    const Tensor& t = args.own(held[i]);
    take(t.scalar_type() == at::kInt && t.is_contiguous());
    return &t;
  }
  int64_t number(PyObject* name) const {
    PyObject* o = get(name);
    int64_t v = 0;
    const bool ok = PyLong_Check(o);
    if (ok) v = PyLong_AsLongLong(o);
    Py_DECREF(o);
    if (PyErr_Occurred()) {
      PyErr_Clear();
      throw NotTaken{};
    }
    take(ok);
    return v;
  }
  int longest() const {
    const int64_t v = number(s_max_query_len);
    take(v >= INT32_MIN && v <= INT32_MAX);
    return (int)v;
  }
};

int mixer_act(const Tensor& t) {
  if (t.scalar_type() == at::kBFloat16) return SW_BF16;
  take(t.scalar_type() == at::kFloat);
  return SW_F32;
}
int hip_act(const Tensor& t) {
  if (t.scalar_type() == at::kHalf) return SW_F16;
  return mixer_act(t);
}
void f32c(const Tensor& t) { take(t.scalar_type() == at::kFloat && t.is_contiguous()); }
int64_t row_stride(const Tensor& t) {
  take(t.dim() == 2 && t.stride(1) == 1);
  return t.stride(0);
}
bool is(const Tensor& t, int64_t a, int64_t b) { return t.dim() == 2 && t.size(0) == a && t.size(1) == b; }
bool is_state(const Tensor& t, int64_t a, int64_t b, int64_t c) {
  return t.dim() == 4 && t.size(1) == a && t.size(2) == b && t.size(3) == c;
}
template <typename T = float> T* ptr(const Tensor& t) { return static_cast<T*>(t.data_ptr()); }
template <typename T = float> T* ptr(const Tensor* t) { return t ? static_cast<T*>(t->data_ptr()) : nullptr; }
Tensor floats(int64_t n, const Tensor& like) { return at::empty({n}, like.options().dtype(at::kFloat)); }

struct Unlocked {                                   // a launch may wait for room in the stream's queue
  PyThreadState* state = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(state); }
};
template <typename F> int unlocked(F f) {
  const Unlocked guard;
  return f();
}
// One call: `body` returns the status or a new object.
template <typename F> PyObject* call(F body) {
  try {
    return body();
  } catch (...) {                                  // also what torch throws: the Python function meets it again
    PyErr_Clear();
    Py_RETURN_NONE;
  }
}
#define STEP_OP(name) PyObject* name(PyObject*, PyObject* const* args, Py_ssize_t nargs)

// ------------------------------------------------------------------------------------------------ Llama path
int cache_dtype(PyObject* o, int act) {
  take(PyUnicode_Check(o));
  if (PyUnicode_CompareWithASCIIString(o, "auto") == 0) return act;
  take(PyUnicode_CompareWithASCIIString(o, "fp8_e5m2") == 0);
  return SW_FP8_E5M2;
}

STEP_OP(reshape_and_cache) {
  return call([&] {
    const Args c(args, nargs, 6);
    take(sw_reshape_and_cache_at != nullptr);
    const Tensor &key = c.tensor(0), &value = c.tensor(1), &kc = c.tensor(2), &vc = c.tensor(3), &slots = c.tensor(4);
    const int act = hip_act(key), cache = cache_dtype(args[5], act);
    take(key.dim() == 3 && value.dim() == 3 && kc.dim() == 5 && slots.scalar_type() == at::kLong);
    const int64_t size = key.size(2);
    take(key.stride(2) == 1 && key.stride(1) == size && value.stride(2) == 1 && value.stride(1) == size);
    void* stream = c.stream();
    return PyLong_FromLong(unlocked([&] {
      return sw_reshape_and_cache_at(ptr<void>(key), ptr<void>(value), ptr<void>(kc), ptr<void>(vc), ptr<int64_t>(slots),
                                     (int)key.size(0), (int)key.size(1), (int)size, (int)kc.size(3), (int)kc.size(4),
                                     key.stride(0), value.stride(0), act, cache, stream);
    }));
  });
}

STEP_OP(paged_attention_v1) {
  return call([&] {
    const Args c(args, nargs, 12);
    take(sw_paged_attention_v1_at != nullptr && args[10] == Py_None);
    const Tensor &out = c.tensor(0), &query = c.tensor(1), &kc = c.tensor(2), &vc = c.tensor(3), &tables = c.tensor(6),
                 &lens = c.tensor(7);
    const int kv_heads = c.i32(4), block_size = c.i32(8), longest = c.i32(9);
    const float scale = c.f32(5);
    take(query.dim() == 3 && kc.dim() >= 2 && tables.dim() == 2 && tables.scalar_type() == at::kInt
         && lens.scalar_type() == at::kInt && (tables.is_contiguous() || tables.stride(1) == 1));
    const int act = hip_act(query), cache = cache_dtype(args[11], act);
    void* stream = c.stream();
    return PyLong_FromLong(unlocked([&] {
      return sw_paged_attention_v1_at(ptr<void>(out), ptr<void>(query), ptr<void>(kc), ptr<void>(vc), (int)query.size(0),
                                      (int)query.size(1), kv_heads, (int)query.size(2), scale, ptr<int32_t>(tables),
                                      ptr<int32_t>(lens), block_size, longest, (int)tables.stride(0), nullptr, query.stride(0),
                                      kc.stride(0), kc.stride(1), act, cache, stream);
    }));
  });
}

STEP_OP(paged_attention_and_cache) {
  return call([&] {
    const Args c(args, nargs, 17);
    take(sw_paged_attention_and_cache_at != nullptr && args[16] == Py_None);
    const Tensor &out = c.tensor(0), &query = c.tensor(4), &key = c.tensor(5), &value = c.tensor(6), &kc = c.tensor(7), &vc = c.tensor(8),
                 &slots = c.tensor(9), &tables = c.tensor(11), &lens = c.tensor(12);
    const Tensor *sums = c.optional(1), *most = c.optional(2), *tmp = c.optional(3);
    const int longest = c.i32(13);
    const float scale = c.f32(10);
    const int act = hip_act(query), cache = cache_dtype(args[14], act), kv_heads = c.i32(15);
    take(query.dim() == 3 && key.dim() == 3 && kc.dim() == 5 && vc.dim() == 4 && kc.is_contiguous() && vc.is_contiguous()
         && slots.scalar_type() == at::kLong && tables.dim() == 2 && tables.scalar_type() == at::kInt && tables.stride(1) == 1
         && lens.scalar_type() == at::kInt && key.scalar_type() == query.scalar_type() && value.scalar_type() == query.scalar_type()
         && out.scalar_type() == query.scalar_type() && value.sizes() == key.sizes() && key.size(1) == kv_heads
         && key.size(2) == query.size(2) && vc.size(3) == kc.size(3));
    for (const Tensor* t : {&query, &key, &value}) take(t->stride(2) == 1 && t->stride(1) == t->size(2));
    void* stream = c.stream();
    return PyLong_FromLong(unlocked([&] {
      return sw_paged_attention_and_cache_at(
          ptr<void>(out), ptr(sums), ptr(most), ptr<void>(tmp), ptr<void>(query), ptr<void>(key), ptr<void>(value), ptr<void>(kc),
          ptr<void>(vc), ptr<int64_t>(slots), (int)key.size(0), (int)kc.size(4), (int)query.size(0), (int)query.size(1), kv_heads,
          (int)query.size(2), scale, ptr<int32_t>(tables), ptr<int32_t>(lens), (int)kc.size(3), longest, (int)tables.stride(0), nullptr,
          query.stride(0), key.stride(0), value.stride(0), kc.stride(0), kc.stride(1), act, cache, stream);
    }));
  });
}

STEP_OP(prefill_attention) {
  return call([&] {
    const Args c(args, nargs, 10);
    take(sw_prefill_attention_at != nullptr && args[8] == Py_None);
    const Tensor &out = c.tensor(0), &q = c.tensor(1), &k = c.tensor(2), &v = c.tensor(3), &starts = c.tensor(4),
                 &lens = c.tensor(5);
    const int longest = c.i32(6), window = args[9] == Py_None ? 0 : c.i32(9);
    const float scale = c.f32(7);
    take(starts.scalar_type() == at::kInt && lens.scalar_type() == at::kInt);
    for (const Tensor* t : {&out, &q, &k, &v}) take(t->dim() == 3 && t->stride(2) == 1 && t->stride(1) == t->size(2));
    const int act = hip_act(q);
    void* stream = c.stream();
    return PyLong_FromLong(unlocked([&] {
      return sw_prefill_attention_at(ptr<void>(out), ptr<void>(q), ptr<void>(k), ptr<void>(v), ptr<int32_t>(starts),
                                     ptr<int32_t>(lens), (int)lens.numel(), longest, (int)q.size(1), (int)k.size(1),
                                     (int)q.size(2), scale, nullptr, q.stride(0), k.stride(0), v.stride(0), out.stride(0), window,
                                     act, stream);
    }));
  });
}

STEP_OP(prefill_attention_and_cache) {
  return call([&] {
    const Args c(args, nargs, 14);
    take(sw_prefill_attention_and_cache_at != nullptr && args[8] == Py_None);
    const Tensor &out = c.tensor(0), &q = c.tensor(1), &k = c.tensor(2), &v = c.tensor(3), &starts = c.tensor(4),
                 &lens = c.tensor(5), &kc = c.tensor(10), &vc = c.tensor(11), &slots = c.tensor(12);
    const int longest = c.i32(6), window = args[9] == Py_None ? 0 : c.i32(9);
    const float scale = c.f32(7);
    take(starts.scalar_type() == at::kInt && lens.scalar_type() == at::kInt && slots.scalar_type() == at::kLong && kc.dim() == 5);
    for (const Tensor* t : {&out, &q, &k, &v}) take(t->dim() == 3 && t->stride(2) == 1 && t->stride(1) == t->size(2));
    const int act = hip_act(q), cache = cache_dtype(args[13], act);
    take(k.scalar_type() == q.scalar_type() && v.scalar_type() == q.scalar_type() && out.scalar_type() == q.scalar_type()
         && v.sizes() == k.sizes() && k.size(2) == q.size(2));
    void* stream = c.stream();
    return PyLong_FromLong(unlocked([&] {
      return sw_prefill_attention_and_cache_at(
          ptr<void>(out), ptr<void>(q), ptr<void>(k), ptr<void>(v), ptr<int32_t>(starts), ptr<int32_t>(lens), (int)lens.numel(), longest,
          (int)q.size(1), (int)k.size(1), (int)q.size(2), scale, nullptr, q.stride(0), k.stride(0), v.stride(0), out.stride(0), window,
          act, ptr<void>(kc), ptr<void>(vc), ptr<int64_t>(slots), (int)k.size(0), (int)kc.size(3), (int)kc.size(4), cache, stream);
    }));
  });
}

// ------------------------------------------------------------------------------------------------ recurrent mixers
STEP_OP(causal_conv) {
  return call([&] {
    const Args c(args, nargs, 7);
    take(swm_causal_conv_at != nullptr);
    const Tensor &out = c.tensor(0), &x = c.tensor(1), &taps = c.tensor(2), &state = c.tensor(3);
    f32c(taps);
    f32c(state);
    const int64_t stride = row_stride(x), rows = x.size(0), channels = x.size(1);
    const bool silu = c.flag(5), residual = c.flag(6);
    const Ragged b(c, args[4], rows);
    take(taps.dim() == 2 && state.dim() == 3);
    const int64_t k = taps.size(1);
    take(is(out, rows, channels) && out.is_contiguous() && taps.size(0) == channels && state.size(1) == k - 1
         && state.size(2) == channels && b.number(s_max_state_slot) < state.size(0));
    const int out_act = mixer_act(out), x_act = mixer_act(x);
    void* stream = c.stream();
    return PyLong_FromLong(unlocked([&] {
      return swm_causal_conv_at(ptr<void>(out), out_act, ptr<void>(x), x_act, stride, ptr(taps), ptr(state),
                                ptr<int32_t>(b.q_start), ptr<int32_t>(b.ctx_len), ptr<int32_t>(b.token_seq),
                                ptr<int32_t>(b.state_slot), rows, (int)channels, (int)k, silu, residual, 1, stream);
    }));
  });
}

STEP_OP(gated_delta) {
  return call([&] {
    const Args c(args, nargs, 13);
    take(swm_gated_delta_at != nullptr);
    const Tensor &out = c.tensor(0), &qkv = c.tensor(1), &beta = c.tensor(2), &decay = c.tensor(3), &dt_bias = c.tensor(4),
                 &a_log = c.tensor(5), &state = c.tensor(6);
    for (const Tensor* t : {&out, &qkv, &dt_bias, &a_log, &state}) f32c(*t);
    take(qkv.dim() == 2);
    const int64_t rows = qkv.size(0);
    const int heads = c.i32(8), kv_heads = c.i32(9), dim = c.i32(10), vdim = c.i32(11);
    const Ragged b(c, args[7], rows);
    take(heads > 0 && dim > 0 && vdim > 0 && qkv.size(1) == 2ll * kv_heads * dim + (int64_t)heads * vdim
         && is(out, rows, (int64_t)heads * vdim) && is(beta, rows, heads) && is(decay, rows, heads)
         && decay.scalar_type() == beta.scalar_type() && dt_bias.numel() == heads && a_log.numel() == heads
         && is_state(state, heads, dim, vdim) && b.number(s_max_state_slot) < state.size(0));
    const int64_t beta_stride = row_stride(beta), decay_stride = row_stride(decay);
    const int act = mixer_act(decay);
    const bool chunked = (args[12] == Py_None ? b.longest() >= 32 : c.flag(12)) && dim <= 224;
    const Tensor work = floats(chunked ? swm_gated_delta_chunked_workspace_floats_at(rows, b.n, heads, dim, vdim)
                                       : rows * heads * (3ll * ((dim + 3) / 4 * 4) + 1), qkv);
    void* stream = c.stream();
    return PyLong_FromLong(unlocked([&] {
      return (chunked ? swm_gated_delta_chunked_at : swm_gated_delta_at)(
          ptr(out), ptr(qkv), ptr<void>(beta), beta_stride, ptr<void>(decay), decay_stride, ptr(dt_bias), ptr(a_log), ptr(state),
          ptr<int32_t>(b.q_start), ptr<int32_t>(b.ctx_len), ptr<int32_t>(b.state_slot), rows, b.n, heads, kv_heads, dim, vdim,
          ptr(work), act, stream);
    }));
  });
}

STEP_OP(head_norm_gate) {
  return call([&] {
    const Args c(args, nargs, 9);
    take(swm_head_norm_gate_act_at != nullptr);
    const Tensor &out = c.tensor(0), &o = c.tensor(1), &gate = c.tensor(2);
    const Tensor* weight = c.optional(3);
    const bool per_head = c.flag(4), silu = c.flag(8);
    const float eps = c.f32(5);
    const int heads = c.i32(6), vdim = c.i32(7);
    f32c(o);
    if (weight) f32c(*weight);
    take(o.dim() == 2);
    const int64_t rows = o.size(0), width = (int64_t)heads * vdim;
    take(is(o, rows, width) && is(gate, rows, width) && is(out, rows, width) && out.is_contiguous()
         && out.scalar_type() == gate.scalar_type() && (!weight || weight->numel() == (per_head ? width : vdim)));
    const int64_t gate_stride = row_stride(gate);
    const int act = mixer_act(out);
    void* stream = c.stream();
    return PyLong_FromLong(unlocked([&] {
      return swm_head_norm_gate_act_at(ptr<void>(out), ptr(o), ptr<void>(gate), gate_stride, ptr(weight), per_head ? vdim : 0,
                                       eps, rows, heads, vdim, silu, act, stream);
    }));
  });
}

STEP_OP(gla) {
  return call([&] {
    const Args c(args, nargs, 13);
    take(swm_gla_at != nullptr);
    const Tensor &out = c.tensor(0), &q = c.tensor(1), &k = c.tensor(2), &v = c.tensor(3), &decay = c.tensor(4),
                 &state = c.tensor(8);
    const Tensor* bias = c.optional(5);
    const float tau = c.f32(6), q_scale = c.f32(7);
    const int heads = c.i32(10), dim = c.i32(11), vdim = c.i32(12);
    f32c(out);
    f32c(state);
    const int64_t stride = row_stride(q), rows = q.size(0), qw = (int64_t)heads * dim, vw = (int64_t)heads * vdim;
    const Ragged b(c, args[9], rows);
    take(is(q, rows, qw) && is(k, rows, qw) && is(v, rows, vw) && row_stride(k) == stride && row_stride(v) == stride
         && k.scalar_type() == q.scalar_type() && v.scalar_type() == q.scalar_type() && is(decay, rows, qw)
         && decay.scalar_type() == q.scalar_type() && is(out, rows, vw) && is_state(state, heads, dim, vdim)
         && b.number(s_max_state_slot) < state.size(0));
    if (bias) {
      f32c(*bias);
      take(bias->numel() == qw);
    }
    const int64_t decay_stride = row_stride(decay);
    const int longest = b.longest(), act = mixer_act(q);
    const int64_t need = swm_gla_workspace_floats_at(rows, b.n, longest, heads, dim, vdim);
    const Tensor work = need > 0 ? floats(need, q) : Tensor();
    void* stream = c.stream();
    return PyLong_FromLong(unlocked([&] {
      return swm_gla_at(ptr(out), ptr<void>(q), ptr<void>(k), ptr<void>(v), stride, ptr<void>(decay), decay_stride, ptr(bias), tau,
                        q_scale, ptr(state), ptr<int32_t>(b.q_start), ptr<int32_t>(b.ctx_len), ptr<int32_t>(b.state_slot), rows,
                        b.n, longest, heads, dim, vdim, need > 0 ? ptr(work) : nullptr, act, stream);
    }));
  });
}

// lightning and retention differ in what q and k are
template <bool ACTED> PyObject* one_decay(PyObject* const* args, Py_ssize_t nargs) {
  return call([&] {
    const Args c(args, nargs, 10);
    take(swm_lightning_at != nullptr);
    const Tensor &out = c.tensor(0), &q = c.tensor(1), &k = c.tensor(2), &v = c.tensor(3), &decay = c.tensor(4),
                 &state = c.tensor(5);
    const int heads = c.i32(7), dim = c.i32(8), vdim = c.i32(9);
    f32c(out);
    f32c(decay);
    f32c(state);
    const int64_t stride = row_stride(q), v_stride = row_stride(v), rows = q.size(0), qw = (int64_t)heads * dim,
                  vw = (int64_t)heads * vdim;
    if (ACTED) {
      take(row_stride(k) == stride && v_stride == stride && k.scalar_type() == q.scalar_type()
           && v.scalar_type() == q.scalar_type());
    } else {
      f32c(q);
      f32c(k);
    }
    const Ragged b(c, args[6], rows);
    take(is(q, rows, qw) && is(k, rows, qw) && is(v, rows, vw) && is(out, rows, vw) && decay.numel() == heads
         && is_state(state, heads, dim, vdim) && b.number(s_max_state_slot) < state.size(0));
    const int longest = b.longest(), act = mixer_act(v);
    const int64_t need = swm_lightning_workspace_floats_at(rows, b.n, longest, heads, dim, vdim);
    const Tensor work = need > 0 ? floats(need, q) : Tensor();
    float* scratch = need > 0 ? ptr(work) : nullptr;
    void* stream = c.stream();
    return PyLong_FromLong(unlocked([&] {
      if constexpr (ACTED)
        return swm_lightning_at(ptr(out), ptr<void>(q), ptr<void>(k), ptr<void>(v), stride, ptr(decay), ptr(state),
                                ptr<int32_t>(b.q_start), ptr<int32_t>(b.ctx_len), ptr<int32_t>(b.state_slot), rows, b.n, longest,
                                heads, dim, vdim, scratch, act, stream);
      else
        return swm_retention_at(ptr(out), ptr(q), ptr(k), qw, ptr<void>(v), v_stride, ptr(decay), ptr(state),
                                ptr<int32_t>(b.q_start), ptr<int32_t>(b.ctx_len), ptr<int32_t>(b.state_slot), rows, b.n, longest,
                                heads, dim, vdim, scratch, act, stream);
    }));
  });
}
STEP_OP(lightning) { return one_decay<true>(args, nargs); }
STEP_OP(retention) { return one_decay<false>(args, nargs); }

// ------------------------------------------------------------------------------------------------ experts
STEP_OP(group_pairs) {
  return call([&]() -> PyObject* {
    const Args c(args, nargs, 2);
    take(swm_group_pairs_at != nullptr);
    const Tensor& chosen = c.tensor(0);
    const int experts = c.i32(1);
    take(chosen.scalar_type() == at::kInt && chosen.is_contiguous() && experts > 0);
    const int64_t pairs = chosen.numel();
    const Tensor order = at::empty({pairs}, chosen.options()), start = at::empty({experts + 1ll}, chosen.options());
    void* stream = c.stream();
    const int status = unlocked([&] {
      return swm_group_pairs_at(ptr<int32_t>(order), ptr<int32_t>(start), ptr<int32_t>(chosen), pairs, experts, stream);
    });
    if (status != 0) return PyLong_FromLong(status);
    PyObject *o = THPVariable_Wrap(order), *s = THPVariable_Wrap(start);
    PyObject* both = o && s ? PyTuple_Pack(2, o, s) : nullptr;
    Py_XDECREF(o);
    Py_XDECREF(s);
    return both;
  });
}

STEP_OP(expert_ffn) {
  return call([&] {
    const Args c(args, nargs, 12);
    take(swm_expert_up_weighted_at != nullptr);
    const Tensor &out = c.tensor(0), &x = c.tensor(1), &up = c.tensor(2), &down = c.tensor(3), &order = c.tensor(4),
                 &start = c.tensor(5);
    const Tensor* weights = c.optional(9);
    const int top = c.i32(6);
    int activation = c.i32(8);
    const float weight = c.f32(7);
    const bool weigh_input = c.flag(11);
    f32c(out);
    take(x.dim() == 2 && up.dim() == 3 && down.dim() == 3);
    const int64_t rows = x.size(0), width = x.size(1), experts = up.size(0);
    int64_t ff = up.size(1);
    float alpha = 1.0f, limit = INFINITY, shift = 0.0f;
    if (args[10] != Py_None) {
      take(PyTuple_CheckExact(args[10]) && PyTuple_GET_SIZE(args[10]) == 3);
      alpha = Args::real(PyTuple_GET_ITEM(args[10], 0));
      limit = Args::real(PyTuple_GET_ITEM(args[10], 1));
      shift = Args::real(PyTuple_GET_ITEM(args[10], 2));
      ff = down.size(2);
      take(up.size(1) == 32 * ((ff + 15) / 16));
      activation = SWM_ACT_CLAMPED_GLU;
    }
    const int64_t pairs = rows * top;
    take(x.is_contiguous() && up.is_contiguous() && down.is_contiguous() && up.scalar_type() == x.scalar_type()
         && down.scalar_type() == x.scalar_type() && up.size(2) == width && is(out, rows, width) && down.size(0) == experts
         && down.size(1) == width && down.size(2) == ff && order.scalar_type() == at::kInt && order.numel() == pairs
         && order.is_contiguous() && start.scalar_type() == at::kInt && start.numel() == experts + 1 && start.is_contiguous());
    if (weights) {
      f32c(*weights);
      take(weights->numel() == pairs);
    }
    const int act = mixer_act(x);
    const Tensor hidden = at::empty({pairs, ff}, x.options());
    void* stream = c.stream();
    const float* on_pairs = ptr(weights);
    return PyLong_FromLong(unlocked([&] {
      const int status = swm_expert_up_weighted_at(ptr<void>(hidden), ptr<void>(x), ptr<void>(up), ptr<int32_t>(order),
                                                   ptr<int32_t>(start), (int)experts, pairs, (int)width, (int)ff, top, activation,
                                                   alpha, limit, shift, weigh_input ? on_pairs : nullptr, act, stream);
      if (status != 0) return status;
      return swm_expert_down_weighted_at(ptr(out), ptr<void>(hidden), ptr<void>(down), ptr<int32_t>(order), ptr<int32_t>(start),
                                         (int)experts, pairs, (int)width, (int)ff, top, weight, weigh_input ? nullptr : on_pairs,
                                         act, stream);
    }));
  });
}

// ------------------------------------------------------------------------------------------------ paged attention of the mixers
STEP_OP(capped_attention) {
  return call([&] {
    const Args c(args, nargs, 16);
    take(swm_masked_attention_at != nullptr && args[3] != Py_None && args[15] == Py_None);
    const Tensor &out = c.tensor(0), &q = c.tensor(1), &kc = c.tensor(2), &vc = c.tensor(3);
    const Tensor* gate = c.optional(4);
    const int heads = c.i32(6), kv_heads = c.i32(7), dim = c.i32(8), vdim = c.i32(9), window = c.i32(12), chunk = c.i32(13);
    const float scale = c.f32(10), cap = c.f32(11);
    const bool plain_sink = PyBool_Check(args[14]);
    const Tensor* sink = plain_sink ? nullptr : &c.tensor(14);
    if (sink) {
      f32c(*sink);
      take(sink->numel() == heads);
    }
    f32c(q);
    take(q.dim() == 2);
    const int64_t rows = q.size(0), vw = (int64_t)heads * vdim;
    Ragged b(c, args[5], rows);
    const Tensor& tables = *b.part(4, s_block_tables);
    const int64_t out_stride = row_stride(out);
    take(tables.dim() == 2 && tables.size(0) == b.n && is(q, rows, (int64_t)heads * dim) && is(out, rows, vw)
         && out.scalar_type() == kc.scalar_type() && kc.is_contiguous() && kc.dim() == 3
         && kc.size(2) >= (int64_t)kv_heads * dim && vc.scalar_type() == out.scalar_type() && vc.is_contiguous() && vc.dim() == 3
         && vc.size(0) == kc.size(0) && vc.size(1) == kc.size(1) && vc.size(2) >= (int64_t)kv_heads * vdim
         && b.number(s_max_pages_used) <= tables.size(1) && b.number(s_max_page_id) < kc.size(0));
    int64_t gate_stride = 0;
    if (gate) {
      take(is(*gate, rows, vw) && gate->scalar_type() == out.scalar_type());
      gate_stride = row_stride(*gate);
    }
    const int longest = b.longest(), act = mixer_act(out), page = (int)kc.size(1), table_width = (int)tables.size(1);
    const int64_t need =
        swm_masked_attention_workspace_floats_at(rows, b.n, longest, heads, kv_heads, vdim, page, table_width, window, chunk);
    const Tensor work = need > 0 ? floats(need, q) : Tensor();
    float* scratch = need > 0 ? ptr(work) : nullptr;
    void* stream = c.stream();
    return PyLong_FromLong(unlocked([&] {
      if (sink)
        return swm_sink_attention_at(ptr<void>(out), out_stride, ptr(q), ptr<void>(kc), ptr<void>(vc), ptr<void>(gate), gate_stride,
                                     ptr(sink), ptr<int32_t>(tables), table_width, ptr<int32_t>(b.q_start),
                                     ptr<int32_t>(b.ctx_len), rows, b.n, longest, heads, kv_heads, dim, vdim, page, scale, cap,
                                     window, chunk, kc.size(2), vc.size(2), scratch, act, stream);
      return swm_masked_attention_at(ptr<void>(out), out_stride, ptr(q), ptr<void>(kc), ptr<void>(vc), ptr<void>(gate), gate_stride,
                                     ptr<int32_t>(tables), table_width, ptr<int32_t>(b.q_start), ptr<int32_t>(b.ctx_len), rows,
                                     b.n, longest, heads, kv_heads, dim, vdim, page, scale, cap, window, chunk,
                                     args[14] == Py_True, kc.size(2), vc.size(2), scratch, act, stream);
    }));
  });
}

// bind({name: address}): entry points of a library that was loaded
PyObject* bind(PyObject*, PyObject* table) {
  if (!PyDict_Check(table)) return PyErr_Format(PyExc_TypeError, "bind: a dict of addresses");
  PyObject *key, *value;
  Py_ssize_t at = 0;
  while (PyDict_Next(table, &at, &key, &value)) {
    void* address = PyLong_AsVoidPtr(value);
    if (address == nullptr && PyErr_Occurred()) return nullptr;
#define BIND(name) \
  if (PyUnicode_CompareWithASCIIString(key, #name) == 0) name##_at = reinterpret_cast<decltype(&::name)>(address);
    STEP_OPS(BIND)
#undef BIND
  }
  Py_RETURN_NONE;
}

#define METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr},
PyMethodDef kMethods[] = {
    METHOD(reshape_and_cache) METHOD(paged_attention_v1) METHOD(prefill_attention) METHOD(causal_conv) METHOD(gated_delta)
    METHOD(prefill_attention_and_cache) METHOD(paged_attention_and_cache)
    METHOD(head_norm_gate) METHOD(gla) METHOD(lightning) METHOD(retention) METHOD(group_pairs) METHOD(expert_ffn)
    METHOD(capped_attention) {"bind", bind, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_step_ops", nullptr, -1, kMethods};

}  // namespace

PyMODINIT_FUNC PyInit__step_ops() {
  PyObject* torch_c = PyImport_ImportModule("torch._C");
  if (torch_c == nullptr) return nullptr;
  g_raw_stream = PyObject_GetAttrString(torch_c, "_cuda_getCurrentRawStream");
  Py_DECREF(torch_c);
  if (g_raw_stream == nullptr) return nullptr;
#define NAME(n) if ((s_##n = PyUnicode_InternFromString(#n)) == nullptr) return nullptr;
  NAME(q_start) NAME(ctx_len) NAME(token_seq) NAME(state_slot) NAME(block_tables) NAME(max_state_slot) NAME(max_query_len)
  NAME(max_pages_used) NAME(max_page_id)
#undef NAME
  PyObject* m = PyModule_Create(&kModule);
  if (m == nullptr) return nullptr;
  PyModule_AddStringConstant(m, "TORCH", STEP_OPS_TORCH);      // _native.py uses no other torch's
  PyModule_AddIntConstant(m, "SW_ABI_VERSION", SW_ABI_VERSION);
  PyModule_AddIntConstant(m, "SWM_ABI_VERSION", SWM_ABI_VERSION);
  return m;
}
