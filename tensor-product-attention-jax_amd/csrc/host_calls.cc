// Host side of the Python operator API: argument checks, output and workspace allocation, and the call into the C ABI,
// as one native call per operator, plus the operator's autograd node.
//
// What bounds it: a decode of one sequence is two kernels of a few microseconds, and the same work written in Python
// (shape checks, three torch allocations, six factor descriptors and an argument structure through ctypes, a stream
// look-up) took 24 us per call, a differentiable call 100 us - longer than the kernels it launches.  Here a call costs
// what its allocations and launches cost.
//
// Every function takes its operands as torch GPU tensors and returns NotImplemented if one of them is something else
// (numpy arrays, CPU tensors): the Python layer then converts them and calls again.  The shape and type rules are those
// of tpa/tpa.py:144-163,474-475; a violated one raises the exception a Python `assert` / `raise` would.
#include <Python.h>
#include <dlfcn.h>

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>

#include <string>
#include <utility>

#include "tpa_abi.h"

namespace {

using at::Tensor;

// ------------------------------------------------------------------------------------------------ the C ABI, by name
#define TPA_CALLS(X)                                                                                             \
  X(tpa_fwd) X(tpa_decode) X(tpa_cache_append) X(tpa_bwd) X(tpa_strerror) X(tpa_fwd_call_workspace_bytes) \
  X(tpa_decode_call_workspace_bytes) X(tpa_cache_append_workspace_bytes) X(tpa_bwd_workspace_bytes)
struct Library {
#define X(name) decltype(&::name) name = nullptr;
  TPA_CALLS(X)
#undef X
} lib;

// ------------------------------------------------------------------------------------------------ errors
PyObject* error_class = nullptr;  // TpaError(function, code, text)

struct Raise {  // a Python exception of a built-in type
  PyObject* type;
  std::string text;
};
struct CallFailed {  // a non-zero return code of the C ABI
  const char* function;
  int code;
};
void check(const char* function, int code) {
  if (code != TPA_OK) throw CallFailed{function, code};
}
std::string sizes_of(const Tensor& t) {
  std::string s = "torch.Size([";
  for (int64_t i = 0; i < t.dim(); ++i) s += (i ? ", " : "") + std::to_string(t.size(i));
  return s + "])";
}
void expect(bool ok, const Tensor& t) {
  if (!ok) throw Raise{PyExc_AssertionError, sizes_of(t)};
}
void set_python_error(const CallFailed& e) {  // with the GIL held
  PyObject* exc = PyObject_CallFunction(error_class, "sis", e.function, e.code, lib.tpa_strerror(e.code));
  if (!exc) return;
  PyErr_SetObject(error_class, exc);
  Py_DECREF(exc);
}

#define BEGIN_CALL HANDLE_TH_ERRORS try {
#define END_CALL                                   \
  }                                                \
  catch (const Raise& e) {                         \
    PyErr_SetString(e.type, e.text.c_str());       \
    return nullptr;                                \
  }                                                \
  catch (const CallFailed& e) {                    \
    set_python_error(e);                           \
    return nullptr;                                \
  }                                                \
  END_HANDLE_TH_ERRORS

struct WithoutGil {
  PyThreadState* state = PyEval_SaveThread();
  ~WithoutGil() { PyEval_RestoreThread(state); }
};

// ------------------------------------------------------------------------------------------------ arguments
// `need` tensors at the front of `args` must be GPU tensors; false: let Python convert them
bool gpu_tensors(PyObject* const* args, int n) {
  for (int i = 0; i < n; ++i)
    if (!THPVariable_Check(args[i]) || !THPVariable_Unpack(args[i]).is_cuda()) return false;
  return true;
}
bool none_or_gpu(PyObject* arg) { return arg == Py_None || gpu_tensors(&arg, 1); }
Tensor tensor_or_none(PyObject* arg) { return arg == Py_None ? Tensor() : THPVariable_Unpack(arg); }
int64_t integer(PyObject* arg) {
  const long long v = PyLong_AsLongLong(arg);
  if (v == -1 && PyErr_Occurred()) throw python_error();
  return v;
}
double real(PyObject* arg) {
  const double v = PyFloat_AsDouble(arg);
  if (v == -1.0 && PyErr_Occurred()) throw python_error();
  return v;
}
void count(const char* name, Py_ssize_t got, Py_ssize_t want) {
  if (got != want) throw Raise{PyExc_TypeError, std::string(name) + ": " + std::to_string(want) + " arguments expected, got " + std::to_string(got)};
}

int dtype_code(at::ScalarType t) {
  if (t == at::kFloat) return TPA_DTYPE_F32;
  if (t == at::kBFloat16) return TPA_DTYPE_BF16;
  throw Raise{PyExc_TypeError, std::string("unsupported dtype ") + c10::toString(t) + ": the kernels take float32 or bfloat16"};
}

// A [b, l, r, x] array whose last dimension is contiguous: `first` .. `first + width` of it
template <typename F>
F factor_of(const Tensor& t, int64_t first = 0) {
  if (t.dim() != 4) throw Raise{PyExc_ValueError, "factor arrays are 4-D [b, l, r, x], got shape " + sizes_of(t)};
  if (t.size(3) > 1 && t.stride(3) != 1) throw Raise{PyExc_ValueError, "the last dimension of a factor array must be contiguous"};
  F f;
  f.ptr = reinterpret_cast<decltype(f.ptr)>(static_cast<char*>(t.data_ptr()) + first * t.element_size());
  f.stride_b = t.stride(0);
  f.stride_l = t.stride(1);
  f.stride_r = t.stride(2);
  return f;
}

bool is_shape(const Tensor& t, std::initializer_list<int64_t> want) { return t.sizes() == at::IntArrayRef(want); }

// int32 [batch, length], one row for all batch entries broadcast (tpa/tpa.py:144-163 vmaps with in_axes=None)
Tensor segment_ids(const Tensor& ids, int64_t batch, int64_t length) {
  if (!ids.defined()) return ids;
  Tensor t = ids.scalar_type() == at::kInt ? ids : ids.to(at::kInt);
  if (t.dim() == 1) t = t.unsqueeze(0).expand({batch, length});
  if (!is_shape(t, {batch, length}))
    throw Raise{PyExc_ValueError, "segment ids must have shape (" + std::to_string(batch) + ", " + std::to_string(length) + "), got " + sizes_of(t)};
  return t.contiguous();
}
Tensor lengths(const Tensor& len, int64_t batch) {
  if (!len.defined()) return len;
  Tensor t = len.scalar_type() == at::kInt ? len.contiguous() : len.to(at::kInt).contiguous();
  if (!is_shape(t, {batch})) throw Raise{PyExc_ValueError, "kv_lengths must have shape (" + std::to_string(batch) + ",), got " + sizes_of(t)};
  return t;
}
const int32_t* ids_ptr(const Tensor& t) { return t.defined() ? static_cast<const int32_t*>(t.data_ptr()) : nullptr; }
float* f32_ptr(const Tensor& t) { return t.defined() ? static_cast<float*>(t.data_ptr()) : nullptr; }

Tensor bytes_on(const at::Device& device, size_t n) { return at::empty({(int64_t)n}, at::TensorOptions().dtype(at::kByte).device(device)); }
void* aligned(const Tensor& t, size_t to) {
  const uintptr_t p = reinterpret_cast<uintptr_t>(t.data_ptr());
  return reinterpret_cast<void*>((p + to - 1) / to * to);
}
void* stream_of(const at::Device& device) { return c10::hip::getCurrentHIPStream(device.index()).stream(); }

// ------------------------------------------------------------------------------------------------ forward
struct FwdCall {
  Tensor qseg, kvseg, kvlen;
  double sm_scale = 1.0;
  int causal = 0, kernel = TPA_KERNEL_AUTO, causal_offset = 0, nomat = 0;
  bool return_lse = true, use_workspace = true;
};

// `a` holds the six factors and the sizes; allocates the outputs and the workspace and makes the call
std::pair<Tensor, Tensor> run_fwd(TpaFwdArgs& a, const FwdCall& c, const at::Device& device, at::ScalarType dtype) {
  a.dtype = dtype_code(dtype);
  const Tensor qseg = segment_ids(c.qseg, a.B, a.lq), kvseg = segment_ids(c.kvseg, a.B, a.lk);
  if (qseg.defined() != kvseg.defined()) throw Raise{PyExc_ValueError, "q_segment_ids and kv_segment_ids must be given together"};
  const Tensor kvlen = lengths(c.kvlen, a.B);
  const auto options = at::TensorOptions().device(device);
  Tensor o = at::empty({a.B, a.lq, a.H, a.dv}, options.dtype(dtype)), lse, ws;
  if (c.return_lse) lse = at::empty({a.B, a.H, a.lq}, options.dtype(at::kFloat));
  a.q_segment_ids = ids_ptr(qseg);
  a.kv_segment_ids = ids_ptr(kvseg);
  a.kv_lengths = ids_ptr(kvlen);
  a.o = o.data_ptr();
  a.lse = f32_ptr(lse);
  a.sm_scale = (float)c.sm_scale;
  a.causal = c.causal;
  a.kernel = c.kernel;
  a.causal_offset = c.causal_offset;
  a.nomat = c.nomat;
  // the workspace with which the library can pick its fastest kernel (nomat: the split partials, required)
  const size_t need = c.use_workspace || c.nomat ? lib.tpa_fwd_call_workspace_bytes(&a) : 0;
  if (need) {
    try {
      ws = bytes_on(device, need + 256);
    } catch (const c10::OutOfMemoryError&) {
      if (c.nomat) throw;  // otherwise it is optional: on a card too full for it the kernels that take none serve the call
    }
  }
  if (ws.defined()) {
    a.workspace = aligned(ws, 256);
    a.workspace_bytes = need;
  }
  check("tpa_fwd", lib.tpa_fwd(&a, stream_of(device)));
  return {o, lse};
}

void check_dtypes(const Tensor* t, const char* const* names, int n) {
  for (int i = 1; i < n; ++i)
    if (t[i].scalar_type() != t[0].scalar_type())
      throw Raise{PyExc_TypeError, std::string(names[i]) + " has dtype " + c10::toString(t[i].scalar_type()) + ", expected " + c10::toString(t[0].scalar_type())};
}

// q[b, lq, rq, h + dk], k[b, lk, rk, h + dk], v[b, lk, rk, h + dv] of one type: what the operator and its gradient take
void check_concatenated(const Tensor& q, const Tensor& k, const Tensor& v, int64_t h) {
  if (q.dim() != 4 || k.dim() != 4 || v.dim() != 4) throw Raise{PyExc_ValueError, "q, k, v must be [b, l, r, h + d]"};
  // rank and length of the keys are read from v (tpa/tpa.py:474-475)
  expect(is_shape(k, {q.size(0), v.size(1), v.size(2), q.size(3)}), k);
  expect(v.size(0) == q.size(0), v);
  if (!(0 < h && h < q.size(3) && h < v.size(3)))
    throw Raise{PyExc_AssertionError, "num_heads = " + std::to_string(h) + ", " + sizes_of(q) + ", " + sizes_of(v)};
  const Tensor three[3] = {q, k, v};
  static const char* const names[3] = {"q", "k", "v"};
  check_dtypes(three, names, 3);
}

void unpack_six(PyObject* const* args, Tensor* t) {
  static const char* const names[6] = {"qa", "qb", "ka", "kb", "va", "vb"};
  for (int i = 0; i < 6; ++i) t[i] = THPVariable_Unpack(args[i]);
  check_dtypes(t, names, 6);
  for (int i = 0; i < 6; ++i)
    if (t[i].dim() != 4) throw Raise{PyExc_ValueError, "factor arrays are 4-D [b, l, r, x], got shape " + sizes_of(t[i])};
}

// the six factors and the sizes of a problem whose keys are not paged
template <typename Args>
void describe(const Tensor* t, Args& a) {
  a.B = (int)t[0].size(0); a.lq = (int)t[0].size(1); a.rq = (int)t[0].size(2); a.H = (int)t[0].size(3);
  a.lk = (int)t[5].size(1); a.rk = (int)t[5].size(2); a.dv = (int)t[5].size(3); a.dk = (int)t[1].size(3);
  // shape rules of tpa/tpa.py:474-475: k and v share length and rank, q and k share h + dk
  expect(is_shape(t[1], {a.B, a.lq, a.rq, a.dk}), t[1]);
  expect(is_shape(t[2], {a.B, a.lk, a.rk, a.H}), t[2]);
  expect(is_shape(t[3], {a.B, a.lk, a.rk, a.dk}), t[3]);
  expect(is_shape(t[4], {a.B, a.lk, a.rk, a.H}), t[4]);
  expect(t[5].size(0) == a.B, t[5]);
  a.qa = factor_of<TpaFactor>(t[0]); a.qb = factor_of<TpaFactor>(t[1]);
  a.ka = factor_of<TpaFactor>(t[2]); a.kb = factor_of<TpaFactor>(t[3]);
  a.va = factor_of<TpaFactor>(t[4]); a.vb = factor_of<TpaFactor>(t[5]);
}

PyObject* pair(std::pair<Tensor, Tensor>&& r) {
  PyObject* out = PyTuple_New(2);
  if (!out) throw python_error();
  PyTuple_SET_ITEM(out, 0, THPVariable_Wrap(std::move(r.first)));
  if (r.second.defined()) {
    PyTuple_SET_ITEM(out, 1, THPVariable_Wrap(std::move(r.second)));
  } else {
    Py_INCREF(Py_None);
    PyTuple_SET_ITEM(out, 1, Py_None);
  }
  return out;
}

// factors(qa, qb, ka, kb, va, vb, q_segment_ids, kv_segment_ids, kv_lengths, sm_scale, causal, kernel, return_lse,
//         use_workspace, causal_offset, nomat)
PyObject* factors(PyObject*, PyObject* const* args, Py_ssize_t n) {
  BEGIN_CALL
  count("factors", n, 16);
  if (!gpu_tensors(args, 6) || !none_or_gpu(args[6]) || !none_or_gpu(args[7]) || !none_or_gpu(args[8])) Py_RETURN_NOTIMPLEMENTED;
  Tensor t[6];
  unpack_six(args, t);
  TpaFwdArgs a{};
  FwdCall c;
  c.qseg = tensor_or_none(args[6]); c.kvseg = tensor_or_none(args[7]); c.kvlen = tensor_or_none(args[8]);
  c.sm_scale = real(args[9]);
  c.causal = (int)integer(args[10]); c.kernel = (int)integer(args[11]);
  c.return_lse = integer(args[12]); c.use_workspace = integer(args[13]);
  c.causal_offset = (int)integer(args[14]); c.nomat = (int)integer(args[15]);
  describe(t, a);
  std::pair<Tensor, Tensor> r;
  {
    WithoutGil free;
    const c10::DeviceGuard guard(t[0].device());
    r = run_fwd(a, c, t[0].device(), t[0].scalar_type());
  }
  return pair(std::move(r));
  END_CALL
}

// ------------------------------------------------------------------------------------------------ decode
// decode(qa, qb, ka, kb, va, vb, kv_lengths, page_table, workspace, sm_scale, num_splits, kernel, causal, causal_offset)
PyObject* decode(PyObject*, PyObject* const* args, Py_ssize_t n) {
  BEGIN_CALL
  count("decode", n, 14);
  if (!gpu_tensors(args, 6) || !none_or_gpu(args[6]) || !none_or_gpu(args[7]) || !none_or_gpu(args[8])) Py_RETURN_NOTIMPLEMENTED;
  Tensor t[6];
  unpack_six(args, t);
  TpaFwdArgs a{};
  Tensor pages = tensor_or_none(args[7]), ws = tensor_or_none(args[8]);
  if (!pages.defined()) {
    describe(t, a);
  } else {
    // page pools [pages, page_size, rk, x]; the logical cache length is pages_per_seq * page_size
    a.B = (int)t[0].size(0); a.lq = (int)t[0].size(1); a.rq = (int)t[0].size(2); a.H = (int)t[0].size(3);
    a.rk = (int)t[5].size(2); a.dv = (int)t[5].size(3); a.dk = (int)t[1].size(3);
    const int64_t npages = t[5].size(0), page = t[5].size(1);
    if (pages.scalar_type() != at::kInt) pages = pages.to(at::kInt);
    pages = pages.contiguous();
    expect(pages.dim() == 2 && pages.size(0) == a.B, pages);
    expect(is_shape(t[1], {a.B, a.lq, a.rq, a.dk}), t[1]);
    expect(is_shape(t[3], {npages, page, a.rk, a.dk}), t[3]);
    expect(is_shape(t[2], {npages, page, a.rk, a.H}), t[2]);
    expect(is_shape(t[4], {npages, page, a.rk, a.H}), t[4]);
    a.page_table = ids_ptr(pages);
    a.page_size = (int)page;
    a.pages_per_seq = (int)pages.size(1);
    a.lk = a.pages_per_seq * a.page_size;
    a.qa = factor_of<TpaFactor>(t[0]); a.qb = factor_of<TpaFactor>(t[1]);
    a.ka = factor_of<TpaFactor>(t[2]); a.kb = factor_of<TpaFactor>(t[3]);
    a.va = factor_of<TpaFactor>(t[4]); a.vb = factor_of<TpaFactor>(t[5]);
  }
  a.dtype = dtype_code(t[0].scalar_type());
  a.sm_scale = (float)real(args[9]);
  a.num_splits = (int)integer(args[10]);
  a.kernel = (int)integer(args[11]);
  a.causal = (int)integer(args[12]);
  a.causal_offset = (int)integer(args[13]);
  std::pair<Tensor, Tensor> r;
  {
    WithoutGil free;
    const at::Device device = t[0].device();
    const c10::DeviceGuard guard(device);
    const Tensor kvlen = lengths(tensor_or_none(args[6]), a.B);
    a.kv_lengths = ids_ptr(kvlen);
    const auto options = at::TensorOptions().device(device);
    if (!ws.defined()) ws = bytes_on(device, std::max<size_t>(lib.tpa_decode_call_workspace_bytes(&a), 16));
    r.first = at::empty({a.B, a.lq, a.H, a.dv}, options.dtype(t[0].scalar_type()));
    r.second = at::empty({a.B, a.H, a.lq}, options.dtype(at::kFloat));
    a.workspace = ws.data_ptr();
    a.workspace_bytes = ws.numel() * ws.element_size();
    a.o = r.first.data_ptr();
    a.lse = f32_ptr(r.second);
    check("tpa_decode", lib.tpa_decode(&a, stream_of(device)));
  }
  return pair(std::move(r));
  END_CALL
}

// ------------------------------------------------------------------------------------------------ cache append
// append(x, w, rope_cos, rope_sin, ka, kb, va, vb, kv_lengths, positions, page_table, workspace, rank_q, kernel, use_workspace)
PyObject* append(PyObject*, PyObject* const* args, Py_ssize_t n) {
  BEGIN_CALL
  count("append", n, 15);
  if (!gpu_tensors(args, 8)) Py_RETURN_NOTIMPLEMENTED;
  for (int i = 8; i < 12; ++i)
    if (!none_or_gpu(args[i])) Py_RETURN_NOTIMPLEMENTED;
  static const char* const names[6] = {"x", "w", "ka", "kb", "va", "vb"};
  Tensor t[6] = {THPVariable_Unpack(args[0]), THPVariable_Unpack(args[1]), THPVariable_Unpack(args[4]),
                 THPVariable_Unpack(args[5]), THPVariable_Unpack(args[6]), THPVariable_Unpack(args[7])};
  check_dtypes(t, names, 6);
  Tensor x = t[0], w = t[1], cos = THPVariable_Unpack(args[2]), sin = THPVariable_Unpack(args[3]);
  const Tensor &ka = t[2], &kb = t[3], &va = t[4], &vb = t[5];
  if (x.dim() != 3) throw Raise{PyExc_ValueError, "x is [b, n, d_model], got shape " + sizes_of(x)};
  TpaAppendArgs a{};
  a.B = (int)x.size(0); a.n = (int)x.size(1); a.d_model = (int)x.size(2);
  a.ka = factor_of<TpaFactor>(ka); a.kb = factor_of<TpaFactor>(kb); a.va = factor_of<TpaFactor>(va); a.vb = factor_of<TpaFactor>(vb);
  a.rk = (int)ka.size(2); a.H = (int)ka.size(3); a.D = (int)kb.size(3); a.rq = (int)integer(args[12]);
  a.dtype = dtype_code(x.scalar_type());
  a.kernel = (int)integer(args[13]);
  (void)integer(args[14]);  // use_workspace: no append kernel takes scratch memory any more
  expect(is_shape(w, {(int64_t)(a.rq + 2 * a.rk) * (a.H + a.D), a.d_model}), w);
  expect(kb.sizes().slice(0, 3) == ka.sizes().slice(0, 3) && va.sizes() == ka.sizes() && vb.sizes() == kb.sizes(), kb);
  expect(cos.sizes() == sin.sizes() && cos.dim() == 2 && cos.size(1) == a.D / 2, cos);
  a.rope_len = (int)cos.size(0);
  Tensor pages = tensor_or_none(args[10]), pos = tensor_or_none(args[9]), ws = tensor_or_none(args[11]), qa, qb, new_len;
  {
    WithoutGil free;
    const at::Device device = x.device();
    const c10::DeviceGuard guard(device);
    if (!pages.defined()) {
      expect(ka.size(0) == a.B, ka);
      a.cache_len = (int)ka.size(1);
    } else {
      if (pages.scalar_type() != at::kInt) pages = pages.to(at::kInt);
      pages = pages.contiguous();
      expect(pages.dim() == 2 && pages.size(0) == a.B, pages);
      a.page_table = ids_ptr(pages);
      a.page_size = (int)ka.size(1);
      a.pages_per_seq = (int)pages.size(1);
      a.cache_len = a.pages_per_seq * a.page_size;
    }
    const Tensor kvlen = lengths(tensor_or_none(args[8]), a.B);
    if (pos.defined()) {
      pos = pos.scalar_type() == at::kInt ? pos.contiguous() : pos.to(at::kInt).contiguous();
      expect(is_shape(pos, {a.B, a.n}), pos);
    }
    x = x.contiguous();
    w = w.contiguous();
    cos = cos.to(at::kFloat).contiguous();
    sin = sin.to(at::kFloat).contiguous();
    const auto options = at::TensorOptions().device(device);
    qa = at::empty({a.B, a.n, a.rq, a.H}, options.dtype(x.scalar_type()));
    qb = at::empty({a.B, a.n, a.rq, a.D}, options.dtype(x.scalar_type()));
    new_len = at::empty({a.B}, options.dtype(at::kInt));
    if (ws.defined()) {
      a.workspace = aligned(ws, 16);
      a.workspace_bytes = ws.numel() * ws.element_size() - (static_cast<char*>(a.workspace) - static_cast<char*>(ws.data_ptr()));
    }
    a.x = x.data_ptr(); a.w = w.data_ptr();
    a.rope_cos = f32_ptr(cos); a.rope_sin = f32_ptr(sin);
    a.positions = ids_ptr(pos); a.kv_lengths = ids_ptr(kvlen); a.new_kv_lengths = static_cast<int32_t*>(new_len.data_ptr());
    a.qa = factor_of<TpaFactor>(qa); a.qb = factor_of<TpaFactor>(qb);
    check("tpa_cache_append", lib.tpa_cache_append(&a, stream_of(device)));
  }
  PyObject* out = PyTuple_New(3);
  if (!out) throw python_error();
  PyTuple_SET_ITEM(out, 0, THPVariable_Wrap(std::move(qa)));
  PyTuple_SET_ITEM(out, 1, THPVariable_Wrap(std::move(qb)));
  PyTuple_SET_ITEM(out, 2, THPVariable_Wrap(std::move(new_len)));
  return out;
  END_CALL
}

// ------------------------------------------------------------------------------------------------ backward
// Gradients of the six factors into concatenated arrays dq, dk, dv of the inputs' type (tpa/tpa.py:960-962); `lse` is [b, h, lq].
struct BwdCall {
  Tensor q, k, v, qseg, kvseg, o, lse, d_o;
  int64_t heads = 0;
  double sm_scale = 1.0;
  int causal = 0, causal_offset = 0;
};

void run_bwd(const BwdCall& c, Tensor* grads) {
  const at::Device device = c.q.device();
  const c10::DeviceGuard guard(device);
  const at::ScalarType dtype = c.q.scalar_type();
  const int64_t h = c.heads;
  TpaBwdArgs a{};
  a.B = (int)c.q.size(0); a.lq = (int)c.q.size(1); a.rq = (int)c.q.size(2); a.H = (int)h; a.dk = (int)(c.q.size(3) - h);
  a.lk = (int)c.v.size(1); a.rk = (int)c.v.size(2); a.dv = (int)(c.v.size(3) - h);
  a.qa = factor_of<TpaFactor>(c.q); a.qb = factor_of<TpaFactor>(c.q, h);
  a.ka = factor_of<TpaFactor>(c.k); a.kb = factor_of<TpaFactor>(c.k, h);
  a.va = factor_of<TpaFactor>(c.v); a.vb = factor_of<TpaFactor>(c.v, h);
  a.dtype = dtype_code(dtype);
  const Tensor qseg = segment_ids(c.qseg, a.B, a.lq), kvseg = segment_ids(c.kvseg, a.B, a.lk);
  const Tensor o = c.o.to(dtype).contiguous(), d_o = c.d_o.to(dtype).contiguous(), lse = c.lse.to(at::kFloat).contiguous();
  expect(is_shape(o, {a.B, a.lq, a.H, a.dv}), o);
  expect(is_shape(d_o, {a.B, a.lq, a.H, a.dv}), d_o);
  expect(is_shape(lse, {a.B, a.H, a.lq}), lse);
  const Tensor* in[3] = {&c.q, &c.k, &c.v};
  for (int i = 0; i < 3; ++i) grads[i] = at::empty(in[i]->sizes(), at::TensorOptions().device(device).dtype(dtype));
  a.dqa = factor_of<TpaGrad>(grads[0]); a.dqb = factor_of<TpaGrad>(grads[0], h);
  a.dka = factor_of<TpaGrad>(grads[1]); a.dkb = factor_of<TpaGrad>(grads[1], h);
  a.dva = factor_of<TpaGrad>(grads[2]); a.dvb = factor_of<TpaGrad>(grads[2], h);
  a.q_segment_ids = ids_ptr(qseg);
  a.kv_segment_ids = ids_ptr(kvseg);
  a.o = o.data_ptr();
  a.lse = f32_ptr(lse);
  a.d_o = d_o.data_ptr();
  a.sm_scale = (float)c.sm_scale;
  a.causal = c.causal;
  a.causal_offset = c.causal_offset;
  a.grad_dtype = a.dtype;
  const size_t need = lib.tpa_bwd_workspace_bytes(a.B, a.lq, a.lk, a.H, a.dk, a.dv);
  const Tensor ws = bytes_on(device, need + 256);
  a.workspace = aligned(ws, 256);
  a.workspace_bytes = need;
  check("tpa_bwd", lib.tpa_bwd(&a, stream_of(device)));
}

// backward(q, k, v, q_segment_ids, kv_segment_ids, o, lse, do, num_heads, sm_scale, causal, causal_offset)
PyObject* backward(PyObject*, PyObject* const* args, Py_ssize_t n) {
  BEGIN_CALL
  count("backward", n, 12);
  if (!gpu_tensors(args, 3) || !gpu_tensors(args + 5, 3) || !none_or_gpu(args[3]) || !none_or_gpu(args[4])) Py_RETURN_NOTIMPLEMENTED;
  BwdCall c;
  c.q = THPVariable_Unpack(args[0]); c.k = THPVariable_Unpack(args[1]); c.v = THPVariable_Unpack(args[2]);
  c.qseg = tensor_or_none(args[3]); c.kvseg = tensor_or_none(args[4]);
  c.o = THPVariable_Unpack(args[5]); c.lse = THPVariable_Unpack(args[6]); c.d_o = THPVariable_Unpack(args[7]);
  c.heads = integer(args[8]);
  check_concatenated(c.q, c.k, c.v, c.heads);
  c.sm_scale = real(args[9]);
  c.causal = (int)integer(args[10]); c.causal_offset = (int)integer(args[11]);
  Tensor grads[3];
  {
    WithoutGil free;
    const at::AutoGradMode no_grad(false);
    run_bwd(c, grads);
  }
  PyObject* out = PyTuple_New(3);
  if (!out) throw python_error();
  for (int i = 0; i < 3; ++i) PyTuple_SET_ITEM(out, i, THPVariable_Wrap(std::move(grads[i])));
  return out;
  END_CALL
}

// ------------------------------------------------------------------------------------------------ the operator
// tpa() on concatenated q[b, lq, rq, h + dk], k[b, lk, rk, h + dk], v[b, lk, rk, h + dv]; the vjp registered for it is
// tpa/tpa.py:217's.
std::pair<Tensor, Tensor> run_concat(const Tensor& q, const Tensor& k, const Tensor& v, int64_t h, const FwdCall& c) {
  const c10::DeviceGuard guard(q.device());
  TpaFwdArgs a{};
  a.B = (int)q.size(0); a.lq = (int)q.size(1); a.rq = (int)q.size(2); a.H = (int)h; a.dk = (int)(q.size(3) - h);
  a.lk = (int)v.size(1); a.rk = (int)v.size(2); a.dv = (int)(v.size(3) - h);
  a.qa = factor_of<TpaFactor>(q); a.qb = factor_of<TpaFactor>(q, h);
  a.ka = factor_of<TpaFactor>(k); a.kb = factor_of<TpaFactor>(k, h);
  a.va = factor_of<TpaFactor>(v); a.vb = factor_of<TpaFactor>(v, h);
  return run_fwd(a, c, q.device(), q.scalar_type());
}

struct Operator : torch::autograd::Function<Operator> {
  static torch::autograd::variable_list forward(torch::autograd::AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v,
                                                int64_t h, const FwdCall& c) {
    auto [o, lse] = run_concat(q, k, v, h, c);
    ctx->mark_non_differentiable({lse});
    ctx->set_materialize_grads(false);
    ctx->save_for_backward({q, k, v, o, lse});
    ctx->saved_data["call"] = c10::IValue(std::make_tuple(h, c.qseg, c.kvseg, c.sm_scale, (int64_t)c.causal, (int64_t)c.causal_offset));
    return {o, lse};
  }
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, torch::autograd::variable_list d_out) {
    torch::autograd::variable_list out(5);
    if (!d_out[0].defined()) return out;
    const auto saved = ctx->get_saved_variables();
    const auto call = ctx->saved_data["call"].toTuple();
    const auto& e = call->elements();
    BwdCall b;
    b.q = saved[0]; b.k = saved[1]; b.v = saved[2]; b.o = saved[3]; b.lse = saved[4];
    b.d_o = d_out[0];
    b.heads = e[0].toInt();
    b.qseg = e[1].toTensor(); b.kvseg = e[2].toTensor();
    b.sm_scale = e[3].toDouble();
    b.causal = (int)e[4].toInt(); b.causal_offset = (int)e[5].toInt();
    try {
      run_bwd(b, out.data());
    } catch (const CallFailed& f) {  // an engine thread: hand the Python exception to the thread that asked
      PyGILState_STATE gil = PyGILState_Ensure();
      set_python_error(f);
      python_error e2;
      e2.persist();
      PyGILState_Release(gil);
      throw e2;
    } catch (const Raise& f) {
      TORCH_CHECK(false, f.text);
    }
    return out;
  }
};

// tpa(q, k, v, q_segment_ids, kv_segment_ids, num_heads, sm_scale, causal, kernel, use_workspace, causal_offset, nomat)
PyObject* tpa(PyObject*, PyObject* const* args, Py_ssize_t n) {
  BEGIN_CALL
  count("tpa", n, 12);
  if (!gpu_tensors(args, 3) || !none_or_gpu(args[3]) || !none_or_gpu(args[4])) Py_RETURN_NOTIMPLEMENTED;
  const Tensor q = THPVariable_Unpack(args[0]), k = THPVariable_Unpack(args[1]), v = THPVariable_Unpack(args[2]);
  const int64_t h = integer(args[5]);
  check_concatenated(q, k, v, h);
  // a dual tensor need not ask for gradients, so the autograd node below, which refuses a tangent, may never see it
  for (const Tensor* t : {&q, &k, &v})
    if (t->_fw_grad(/*level=*/0).defined())
      throw Raise{PyExc_NotImplementedError, "tpa has no forward-mode derivative: an input carries a tangent"};
  FwdCall c;
  c.qseg = tensor_or_none(args[3]); c.kvseg = tensor_or_none(args[4]);
  c.sm_scale = real(args[6]);
  c.causal = (int)integer(args[7]); c.kernel = (int)integer(args[8]);
  c.use_workspace = integer(args[9]);
  c.causal_offset = (int)integer(args[10]); c.nomat = (int)integer(args[11]);
  std::pair<Tensor, Tensor> r;
  {
    WithoutGil free;
    if (at::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad())) {
      auto out = Operator::apply(q, k, v, h, c);
      r = {out[0], out[1]};
    } else {
      r = run_concat(q, k, v, h, c);
    }
  }
  return pair(std::move(r));
  END_CALL
}

// ------------------------------------------------------------------------------------------------ module
// bind(path of libtpa_gfx950.so, TpaError)
PyObject* bind(PyObject*, PyObject* args) {
  const char* path;
  PyObject* cls;
  if (!PyArg_ParseTuple(args, "sO", &path, &cls)) return nullptr;
  void* h = dlopen(path, RTLD_NOW | RTLD_LOCAL);
  if (!h) {
    PyErr_SetString(PyExc_RuntimeError, dlerror());
    return nullptr;
  }
#define X(name)                                                                           \
  lib.name = reinterpret_cast<decltype(lib.name)>(dlsym(h, #name));                       \
  if (!lib.name) {                                                                        \
    PyErr_SetString(PyExc_RuntimeError, "the library does not export " #name);            \
    return nullptr;                                                                       \
  }
  TPA_CALLS(X)
#undef X
  Py_INCREF(cls);
  error_class = cls;
  Py_RETURN_NONE;
}

#define FAST(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {{"bind", bind, METH_VARARGS, nullptr}, FAST(factors), FAST(decode), FAST(append), FAST(backward), FAST(tpa), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "tpa_host_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_tpa_host_calls() { return PyModule_Create(&module); }
