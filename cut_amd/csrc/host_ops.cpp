// Host side of the operators that programs launch one by one (cut_amd/ops.py): the checks of their tensors, the outputs and
// scratch they allocate and the C-ABI call, as one native call each.  In Python, with the call through ctypes, that was 4 to 9 us
// of host time in front of launches that take 2.2 us to issue and often less to run (a decode step of the two-layer test model
// launched operator by operator 107 us -> 68).  Nothing is kept from one call to the next.
//
// Every function takes the positional arguments of the Python function of its name and raises what that raised.
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ops/empty.h>
#include <c10/hip/HIPStream.h>

#include <cstring>

#include "../../include/cut_hip.h"

namespace {

// set once by setup()
PyObject *g_error = nullptr, *g_formats = nullptr, *g_unary = nullptr, *g_binary = nullptr;
PyObject *g_norm_carry = nullptr, *g_rope_append = nullptr, *g_ctypes = nullptr;

struct PyError {};   // a Python exception is set

[[noreturn]] void fail(const char *text) {
  PyErr_SetString(g_error, text);
  throw PyError{};
}
// Other Python threads run while a launch waits (a full queue, the first load of a code object) or memory is allocated: a host
// callback on the stream may need one of them.
struct Released {
  PyThreadState *s = PyEval_SaveThread();
  ~Released() { PyEval_RestoreThread(s); }
};
// a call of the C ABI; its arguments are evaluated before the GIL is given back
template <class... P, class... A> void call(int (*f)(P...), A... args) {
  int rc;
  {
    const Released r;
    rc = f(args...);
  }
  if (rc == 0) return;
  PyErr_Format(g_error, "cut_hip error %d: %s", rc, cuthip_last_error());
  throw PyError{};
}

const at::Tensor &tensor(PyObject *o) {
  if (!THPVariable_Check(o)) {
    PyErr_Format(PyExc_TypeError, "expected a tensor, got %s", Py_TYPE(o)->tp_name);
    throw PyError{};
  }
  return THPVariable_Unpack(o);
}
bool given(PyObject *o) { return o != Py_None; }
int64_t integer(PyObject *o) {
  const int64_t v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) throw PyError{};
  return v;
}
float real(PyObject *o) {
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) throw PyError{};
  return (float)v;
}
bool truth(PyObject *o) {
  const int v = PyObject_IsTrue(o);
  if (v < 0) throw PyError{};
  return v != 0;
}
int lookup(PyObject *table, PyObject *key) {
  PyObject *v = PyDict_GetItemWithError(table, key);
  if (!v) {
    if (!PyErr_Occurred()) PyErr_SetObject(PyExc_KeyError, key);
    throw PyError{};
  }
  return (int)integer(v);
}
int format(PyObject *o) {
  if (!PyUnicode_Check(o)) {   // any number, as int() takes it
    PyObject *number = PyNumber_Long(o);
    if (!number) throw PyError{};
    const int64_t f = PyLong_AsLongLong(number);
    Py_DECREF(number);
    if (f == -1 && PyErr_Occurred()) throw PyError{};
    return f == (int)f ? (int)f : -1;
  }
  PyObject *v = PyDict_GetItemWithError(g_formats, o);
  if (!v) {
    if (!PyErr_Occurred()) PyErr_Format(g_error, "unknown quantization format %R", o);
    throw PyError{};
  }
  return (int)integer(v);
}
void block_of(int f, int64_t &elems, int64_t &bytes) {
  switch (f) {
  case CUTHIP_Q8_0: elems = 32; bytes = 34; return;
  case CUTHIP_Q4_0: elems = 32; bytes = 18; return;
  case CUTHIP_Q4_K: elems = 256; bytes = 144; return;
  case CUTHIP_Q6_K: elems = 256; bytes = 210; return;
  }
  if (PyObject *key = PyLong_FromLong(f)) {
    PyErr_SetObject(PyExc_KeyError, key);
    Py_DECREF(key);
  }
  throw PyError{};
}
// more than any tensor holds for counts that are negative or whose product needs more than 64 bits
int64_t n_bytes(int f, int64_t rows, int64_t cols) {
  int64_t elems, bytes;
  block_of(f, elems, bytes);
  if (cols % elems) {
    PyErr_Format(g_error, "cols (%lld) must be a multiple of the block size %lld", (long long)cols, (long long)elems);
    throw PyError{};
  }
  int64_t n;
  if (rows < 0 || cols < 0 || __builtin_mul_overflow(cols / elems, bytes, &n) || __builtin_mul_overflow(rows, n, &n)) return INT64_MAX;
  return n;
}
bool activation(const at::Tensor &t) { return t.scalar_type() == at::kHalf || t.scalar_type() == at::kFloat; }
int act_dtype(const at::Tensor &t) {
  if (t.scalar_type() == at::kHalf) return CUTHIP_F16;
  if (t.scalar_type() == at::kFloat) return CUTHIP_F32;
  PyErr_Format(g_error, "activations must be float16 or float32, got torch.%s", c10::toString(t.scalar_type()));
  throw PyError{};
}
int f16_or_f32(const at::Tensor &t) { return t.scalar_type() == at::kHalf ? CUTHIP_F16 : CUTHIP_F32; }
const void *ptr(const at::Tensor &t) { return t.const_data_ptr(); }
void *mut(const at::Tensor &t) { return t.data_ptr(); }
void *stream() { return (void *)c10::hip::getCurrentHIPStream().stream(); }
at::Tensor empty(at::IntArrayRef size, at::ScalarType dtype, const at::Tensor &like) {
  const Released r;
  return at::empty(size, at::TensorOptions().dtype(dtype).device(like.device()));
}

// Whether a launch that writes `rows` rows of `width` elements, stride(0) apart, stays inside the tensor's own rows.
bool holds(const at::Tensor &t, int64_t rows, int64_t width) {
  if (t.dim() == 0) return false;
  if (t.dim() == 1) return rows <= 1 && t.size(0) >= width && (t.size(0) <= 1 || t.stride(0) == 1);
  int64_t run = 1;
  for (int64_t d = t.dim() - 1; d > 0; run *= t.size(d--))
    if (t.size(d) != 1 && t.stride(d) != run) return false;
  return t.size(0) >= rows && run >= width;
}
void require(bool ok, const char *what, int64_t rows, int64_t width) {
  if (ok) return;
  PyErr_Format(g_error, "%s %lld rows of %lld", what, (long long)rows, (long long)width);
  throw PyError{};
}

at::Tensor matrix(const at::Tensor &t) {   // [rows, dim]; a row for any other number of dimensions (which may copy)
  if (t.dim() == 2) return t;
  const Released r;
  return t.reshape({1, -1});
}

// The address of a ctypes structure of the given class (null for None).  Anything else is refused as ctypes refuses it: what the
// library reads there are device pointers.
struct Structure {
  Py_buffer b{};
  void *p = nullptr;
  Structure(PyObject *o, PyObject *cls, size_t size) {
    if (o == Py_None) return;
    const int is = PyObject_IsInstance(o, cls);
    if (is < 0) throw PyError{};
    if (!is) refuse(o, cls);
    if (PyObject_GetBuffer(o, &b, PyBUF_SIMPLE)) throw PyError{};
    if ((size_t)b.len < size) {
      PyBuffer_Release(&b);
      refuse(o, cls);
    }
    p = b.buf;
  }
  ~Structure() {
    if (p) PyBuffer_Release(&b);
  }
  Structure(const Structure &) = delete;

 private:
  [[noreturn]] static void refuse(PyObject *o, PyObject *cls) {
    PyObject *r = PyObject_CallMethod(g_ctypes, "byref", "O", o);   // TypeError for what is no ctypes instance
    if (!r) throw PyError{};
    Py_DECREF(r);
    if (PyObject *e = PyObject_GetAttrString(g_ctypes, "ArgumentError")) {
      PyErr_Format(e, "expected an instance of %s, got %s", ((PyTypeObject *)cls)->tp_name, Py_TYPE(o)->tp_name);
      Py_DECREF(e);
    }
    throw PyError{};
  }
};
Structure norm_carry_of(PyObject *o) { return {o, g_norm_carry, sizeof(cuthip_norm_carry_t)}; }
Structure rope_append_of(PyObject *o) { return {o, g_rope_append, sizeof(cuthip_rope_append_t)}; }

PyObject *ref(PyObject *o) {
  Py_INCREF(o);
  return o;
}

struct Op {
  int epilogue = CUTHIP_EPI_NONE, op = 0;
  const void *d = nullptr;
};

PyObject *dequantize(PyObject *const *a) {   // raw, fmt, rows, cols, dtype, out
  const int f = format(a[1]);
  const at::Tensor &raw = tensor(a[0]);
  if (!raw.is_cuda() || raw.element_size() != 1 || !raw.is_contiguous()) fail("dequantize: raw must be a contiguous 1-byte device tensor");
  const int64_t rows = integer(a[2]), cols = integer(a[3]), need = n_bytes(f, rows, cols);
  if (raw.numel() < need) {
    PyErr_Format(g_error, "dequantize: raw holds %lld bytes, %lld needed", (long long)raw.numel(), (long long)need);
    throw PyError{};
  }
  if (!THPDtype_Check(a[4])) fail("dequantize: output dtype must be float32 or float16");
  const at::ScalarType dt = ((THPDtype *)a[4])->scalar_type;
  if (dt != at::kFloat && dt != at::kHalf) fail("dequantize: output dtype must be float32 or float16");
  const at::Tensor out = given(a[5]) ? tensor(a[5]) : empty({rows, cols}, dt, raw);
  require(out.scalar_type() == dt && (out.dim() == 2 ? holds(out, rows, cols) : out.is_contiguous() && out.numel() >= rows * cols),
       "dequantize: out must have the output dtype and contiguous room for", rows, cols);
  call(cuthip_dequant, f, ptr(raw), mut(out), dt == at::kHalf ? CUTHIP_F16 : CUTHIP_F32, (uint32_t)rows, (uint32_t)cols,
                       (uint32_t)(out.dim() == 2 ? out.stride(0) : cols), stream());
  return given(a[5]) ? ref(a[5]) : THPVariable_Wrap(out);
}

// a, w_blocks, fmt, N, K, out_dtype, out, unary, binary, d, variant, workspace, swiglu_pairs
PyObject *matmul_gguf(PyObject *const *p) {
  const int f = format(p[2]);
  const at::Tensor &a = tensor(p[0]), &w = tensor(p[1]);
  const int64_t N = integer(p[3]), K = integer(p[4]);
  if (a.dim() != 1 && a.dim() != 2) fail("matmul: A must be 1D or 2D");
  const bool row = a.dim() == 1;
  const int64_t M = row ? 1 : a.size(0), cols = a.size(row ? 0 : 1), inner = a.stride(row ? 0 : 1), outer = row ? cols * inner : a.stride(0);
  if (cols != K) {
    PyErr_Format(g_error, "matmul: B rows (%lld) must match A cols (%lld)", (long long)K, (long long)cols);
    throw PyError{};
  }
  if (!activation(a) || inner != 1) fail("matmul: A must be float32/float16 with unit inner stride");
  if (w.numel() < n_bytes(f, N, K)) fail("matmul: weight tensor too small for [N, K]");
  const bool pairs = truth(p[12]);
  at::Tensor out;
  if (given(p[6])) {
    out = tensor(p[6]);
  } else {
    if (given(p[5]) && !THPDtype_Check(p[5])) fail("matmul: out_dtype must be a dtype");
    out = empty({M, pairs ? N / 2 : N}, given(p[5]) ? ((THPDtype *)p[5])->scalar_type : a.scalar_type(), a);
  }
  const int dtype = act_dtype(out);
  const int64_t width = pairs ? N / 2 : N;
  require(holds(out, M, width), "matmul: out must have contiguous room for", M, width);
  Op e;
  if (pairs) {
    e.epilogue = CUTHIP_EPI_SWIGLU_PAIRS;
  } else if (given(p[7])) {
    e.epilogue = CUTHIP_EPI_UNARY;
    e.op = lookup(g_unary, p[7]);
  } else if (given(p[8])) {
    const char *bad = "matmul: binary epilogue needs D with the shape, dtype and stride of C";
    if (!given(p[9])) fail(bad);
    const at::Tensor &d = tensor(p[9]);
    if (d.sizes() != out.sizes() || d.scalar_type() != out.scalar_type() || d.stride(0) != out.stride(0) || !holds(d, M, width)) fail(bad);
    e.epilogue = CUTHIP_EPI_BINARY;
    e.op = lookup(g_binary, p[8]);
    e.d = ptr(d);
  }
  const int variant = (int)integer(p[10]);
  if (given(p[11])) {
    const at::Tensor &ws = tensor(p[11]);
    call(cuthip_matmul_gguf_ws, f, ptr(w), ptr(a), f16_or_f32(a), mut(out), dtype, (uint32_t)M, (uint32_t)K, (uint32_t)N,
                                (uint32_t)outer, (uint32_t)out.stride(0), e.epilogue, e.op, e.d, variant, mut(ws),
                                (size_t)(ws.numel() * ws.element_size()), stream());
  } else {
    call(cuthip_matmul_gguf, f, ptr(w), ptr(a), f16_or_f32(a), mut(out), dtype, (uint32_t)M, (uint32_t)K, (uint32_t)N,
                             (uint32_t)outer, (uint32_t)out.stride(0), e.epilogue, e.op, e.d, variant, stream());
  }
  return given(p[6]) ? ref(p[6]) : THPVariable_Wrap(out);
}

PyObject *norm_carry(PyObject *const *p) {   // NormCarry, sumsq_parts, eps, next_norm_weight, next_x16, next_sumsq_parts
  auto at_ = [](PyObject *o, at::ScalarType dtype) -> void * {
    if (!given(o)) return nullptr;
    const at::Tensor &t = tensor(o);
    if (t.scalar_type() != dtype || !t.is_contiguous()) fail("norm_carry: wrong dtype or non-contiguous tensor");
    return mut(t);
  };
  cuthip_norm_carry_t c{};
  c.sumsq_parts = (const float *)at_(p[1], at::kFloat);
  c.eps = real(p[2]);
  c.next_norm_weight = (const float *)at_(p[3], at::kFloat);
  c.next_x16 = (decltype(c.next_x16))at_(p[4], at::kHalf);
  c.next_sumsq_parts = (float *)at_(p[5], at::kFloat);
  PyObject *o = PyObject_CallNoArgs(p[0]);
  if (!o) throw PyError{};
  Py_buffer b;
  if (PyObject_GetBuffer(o, &b, PyBUF_WRITABLE)) {
    Py_DECREF(o);
    throw PyError{};
  }
  std::memcpy(b.buf, &c, sizeof c);
  PyBuffer_Release(&b);
  return o;
}

PyObject *rope_append(PyObject *const *p) {   // RopeAppend, runtime_params, cos_t, sin_t, q_out, k_cache, v_cache, q_dim, head_dim
  const at::Tensor &k = tensor(p[5]), &v = tensor(p[6]), &cos = tensor(p[2]), &q = tensor(p[4]);
  if (k.scalar_type() != at::kHalf || v.scalar_type() != at::kHalf || k.stride(0) != v.stride(0))
    fail("rope_append: caches must be fp16 with one row stride");
  if (!q.is_contiguous() || q.numel() < integer(p[7])) fail("rope_append: q_out must hold q_dim contiguous elements");
  cuthip_rope_append_t r{};
  r.runtime_params = (decltype(r.runtime_params))ptr(tensor(p[1]));
  r.cos_table = (decltype(r.cos_table))ptr(cos);
  r.sin_table = (decltype(r.sin_table))ptr(tensor(p[3]));
  r.q_out = mut(q);
  r.q_out_dtype = act_dtype(q);
  r.k_cache = (decltype(r.k_cache))mut(k);
  r.v_cache = (decltype(r.v_cache))mut(v);
  r.q_dim = (uint32_t)integer(p[7]);
  r.head_dim = (uint32_t)integer(p[8]);
  r.aligned_kv_dim = (uint32_t)k.stride(0);
  r.max_positions = (uint32_t)std::min(k.size(0), cos.size(0));
  PyObject *o = PyObject_CallNoArgs(p[0]);
  if (!o) throw PyError{};
  Py_buffer b;
  if (PyObject_GetBuffer(o, &b, PyBUF_WRITABLE)) {
    Py_DECREF(o);
    throw PyError{};
  }
  std::memcpy(b.buf, &r, sizeof r);
  PyBuffer_Release(&b);
  return o;
}

PyObject *matmul_gguf_carry(PyObject *const *p) {   // a, w_blocks, fmt, N, K, out, carry, binary, d, swiglu_pairs
  const int f = format(p[2]);
  const at::Tensor &a = tensor(p[0]), &w = tensor(p[1]), &out = tensor(p[5]);
  const int64_t N = integer(p[3]), K = integer(p[4]);
  if (a.numel() != K || !activation(a) || !a.is_contiguous() || !out.is_contiguous())
    fail("matmul_carry: A must be a contiguous float32/float16 vector of K elements, out contiguous");
  const bool pairs = truth(p[9]);
  if (w.numel() < n_bytes(f, N, K) || out.numel() != (pairs ? N / 2 : N)) fail("matmul_carry: weight tensor too small or output of the wrong size");
  Op e;
  if (pairs) {
    e.epilogue = CUTHIP_EPI_SWIGLU_PAIRS;
  } else if (given(p[7])) {
    const char *bad = "matmul_carry: binary epilogue needs D with the size and dtype of C";
    if (!given(p[8])) fail(bad);
    const at::Tensor &d = tensor(p[8]);
    if (d.numel() != N || d.scalar_type() != out.scalar_type()) fail(bad);
    e.epilogue = CUTHIP_EPI_BINARY;
    e.op = lookup(g_binary, p[7]);
    e.d = ptr(d);
  }
  const Structure carry = norm_carry_of(p[6]);
  call(cuthip_matmul_gguf_carry, f, ptr(w), ptr(a), act_dtype(a), mut(out), act_dtype(out), (uint32_t)K, (uint32_t)N, e.epilogue, e.op,
                                 e.d, (const cuthip_norm_carry_t *)carry.p, stream());
  return ref(p[5]);
}

// a, wa, fmt_a, Na, out_a, wb, fmt_b, Nb, out_b, K, carry, rope
PyObject *matmul_gguf_pair(PyObject *const *p) {
  const int fa = format(p[2]), fb = format(p[6]);
  const at::Tensor &a = tensor(p[0]), &wa = tensor(p[1]), &wb = tensor(p[5]);
  const int64_t Na = integer(p[3]), Nb = integer(p[7]), K = integer(p[9]);
  if (a.numel() != K || !activation(a) || !a.is_contiguous()) fail("matmul_pair: A must be a contiguous float32/float16 vector of K elements");
  if (wa.numel() < n_bytes(fa, Na, K) || wb.numel() < n_bytes(fb, Nb, K)) fail("matmul_pair: weight tensor too small for [N, K]");
  const Structure carry = norm_carry_of(p[10]), rope = rope_append_of(p[11]);
  void *ca = nullptr, *cb = nullptr;
  int cdt = CUTHIP_F32;
  if (!rope.p) {   // (with it the epilogue writes q_out and the caches; the plain outputs are not used)
    const at::Tensor &oa = tensor(p[4]), &ob = tensor(p[8]);
    if (oa.scalar_type() != ob.scalar_type() || oa.numel() != Na || ob.numel() != Nb || !oa.is_contiguous() || !ob.is_contiguous())
      fail("matmul_pair: outputs must be contiguous [Na] and [Nb] of one dtype");
    ca = mut(oa);
    cb = mut(ob);
    cdt = act_dtype(oa);
  }
  call(cuthip_matmul_gguf_pair, fa, ptr(wa), (uint32_t)Na, ca, fb, ptr(wb), (uint32_t)Nb, cb, ptr(a), act_dtype(a), cdt, (uint32_t)K,
                                (const cuthip_norm_carry_t *)carry.p, (const cuthip_rope_append_t *)rope.p, stream());
  return ref(Py_None);
}

PyObject *rmsnorm(PyObject *const *p) {   // x, weight, eps, out, out_dtype
  const at::Tensor &x = tensor(p[0]), &w = tensor(p[1]);
  const at::Tensor x2 = matrix(x);
  if (w.scalar_type() != at::kFloat || w.numel() != x2.size(1) || x2.stride(1) != 1) fail("rmsnorm: weight must be fp32 [dim] and x rows contiguous");
  const float eps = real(p[2]);
  if (given(p[4]) && !THPDtype_Check(p[4])) fail("rmsnorm: out_dtype must be a dtype");
  // rows of x and out lie equally far apart
  const int64_t rows = x2.size(0), dim = x2.size(1), stride = x2.stride(0);
  at::Tensor out;
  if (given(p[3])) {
    out = tensor(p[3]);
    require((holds(out, rows, dim) && (rows <= 1 || out.stride(0) == stride)) || (out.is_contiguous() && out.numel() >= (rows - 1) * stride + dim),
         "rmsnorm: out must have contiguous room, as far apart as the rows of x, for", rows, dim);
  } else {
    const at::ScalarType dtype = given(p[4]) ? ((THPDtype *)p[4])->scalar_type : x.scalar_type();
    out = rows > 1 && stride > dim ? empty({rows, stride}, dtype, x).slice(1, 0, dim) : empty(x2.sizes(), dtype, x);
  }
  call(cuthip_rmsnorm, ptr(x2), act_dtype(x2), (const float *)ptr(w), mut(out), act_dtype(out), (uint32_t)rows, (uint32_t)dim,
                       (uint32_t)stride, eps, stream());
  return given(p[3]) ? ref(p[3]) : THPVariable_Wrap(out);
}

// q, k_cache, v_cache, runtime_params, n_heads, n_kv_heads, head_dim, scale, workspace, out, max_seq_len
PyObject *attn_decode(PyObject *const *p) {
  const at::Tensor &q = tensor(p[0]), &k = tensor(p[1]), &v = tensor(p[2]), &par = tensor(p[3]), &ws = tensor(p[8]), &out = tensor(p[9]);
  const int64_t len = given(p[10]) && truth(p[10]) ? integer(p[10]) : k.size(0);
  require(out.is_contiguous() && out.numel() >= integer(p[4]) * integer(p[6]), "attn_decode: out must have contiguous room for", integer(p[4]), integer(p[6]));
  call(cuthip_attn_decode, ptr(q), act_dtype(q), ptr(k), ptr(v), (const uint32_t *)ptr(par), mut(out), act_dtype(out), (uint32_t)integer(p[4]),
                           (uint32_t)integer(p[5]), (uint32_t)integer(p[6]), (uint32_t)k.stride(0), real(p[7]), (uint32_t)len, mut(ws),
                           (size_t)ws.numel(), stream());
  return ref(p[9]);
}

PyObject *silu_mul(PyObject *const *p) {   // gate_up, out
  const at::Tensor &g = tensor(p[0]), &out = tensor(p[1]);
  if (!out.is_contiguous() || !g.is_contiguous() || g.numel() < 2 * out.numel()) fail("silu_mul: gate_up must hold two contiguous halves of the size of out");
  call(cuthip_silu_mul, ptr(g), act_dtype(g), mut(out), act_dtype(out), (uint32_t)out.numel(), stream());
  return ref(p[1]);
}

// a, w_blocks, fmt, N, K, logits, out_index, carry, pen_tokens, pen_factors, workspace
PyObject *matmul_gguf_argmax(PyObject *const *p) {
  const int f = format(p[2]);
  const at::Tensor &a = tensor(p[0]), &w = tensor(p[1]), &logits = tensor(p[5]), &index = tensor(p[6]);
  const int64_t N = integer(p[3]), K = integer(p[4]);
  if (a.numel() != K || !a.is_contiguous() || logits.numel() != N || !logits.is_contiguous())
    fail("matmul_gguf_argmax: a is a contiguous vector of K elements, logits one of N");
  const void *pt = nullptr, *pf = nullptr;
  uint32_t n = 0;
  if (given(p[8])) {
    const at::Tensor &t = tensor(p[8]), &fac = tensor(p[9]);
    if (t.scalar_type() != at::kInt || fac.scalar_type() != at::kFloat || t.numel() != fac.numel())
      fail("penalised tokens are int32 ids with one fp32 factor each");
    pt = ptr(t);
    pf = ptr(fac);
    n = (uint32_t)t.numel();
  }
  const Structure carry = norm_carry_of(p[7]);
  const at::Tensor ws = given(p[10]) ? tensor(p[10]) : at::Tensor();
  call(cuthip_matmul_gguf_argmax, f, ptr(w), ptr(a), act_dtype(a), mut(logits), act_dtype(logits), (uint32_t)K, (uint32_t)N,
                                  (const cuthip_norm_carry_t *)carry.p, (const int32_t *)pt, (const float *)pf, n,
                                  ws.defined() ? mut(ws) : nullptr, ws.defined() ? (size_t)ws.numel() : 0, (uint32_t *)mut(index), stream());
  return ref(p[6]);
}

PyObject *embedding_rows(PyObject *const *p) {   // w_blocks, fmt, token_ids, n_rows, dim, out
  const at::Tensor &w = tensor(p[0]), &ids = tensor(p[2]), &out = tensor(p[5]);
  const int64_t rows = integer(p[3]), dim = integer(p[4]);
  if ((ids.scalar_type() != at::kInt && ids.scalar_type() != at::kUInt32) || out.stride(-1) != 1 || out.numel() < ids.numel() * dim)
    fail("embedding_rows: token ids are 32-bit integers, out holds one row of dim per id");
  const at::Tensor out2 = out.dim() == 2 ? out : out.view({ids.numel(), -1});
  require(holds(out2, ids.numel(), dim), "embedding_rows: out must have contiguous room for", ids.numel(), dim);
  call(cuthip_embedding_rows, format(p[1]), ptr(w), (const uint32_t *)ptr(ids), (uint32_t)ids.numel(), (uint32_t)rows, (uint32_t)dim, mut(out2),
                              act_dtype(out2), (uint32_t)out2.stride(0), stream());
  return ref(p[5]);
}

// a, b, scales, N, q4, affine, out, unary, binary, d, variant
PyObject *matmul_sep(PyObject *const *p) {
  const at::Tensor &in = tensor(p[0]), &b = tensor(p[1]), &s = tensor(p[2]);
  const at::Tensor a = matrix(in);
  const int64_t M = a.size(0), K = a.size(1), N = integer(p[3]);
  const bool q4 = truth(p[4]), affine = truth(p[5]);
  if (a.scalar_type() != at::kFloat || s.scalar_type() != at::kHalf || b.element_size() != 1 || b.dim() != 2 || s.dim() != 2)
    fail("matmul_sep: a must be fp32, b a 2-D 1-byte tensor and scales a 2-D fp16 tensor");
  const int64_t rows_s = (affine ? 2 : 1) * (K / 32);
  if (b.size(0) != K || s.size(0) != rows_s || b.size(1) < (q4 ? (N + 1) / 2 : N) || s.size(1) < N) {
    PyErr_Format(g_error, "matmul_sep: shapes do not match K = %lld, N = %lld (b (%lld, %lld), scales (%lld, %lld))", (long long)K, (long long)N,
                 (long long)b.size(0), (long long)b.size(1), (long long)s.size(0), (long long)s.size(1));
    throw PyError{};
  }
  const at::Tensor out = given(p[6]) ? tensor(p[6]) : empty({M, N}, at::kFloat, in);
  require(out.scalar_type() == at::kFloat && holds(out, M, N), "matmul_sep: out must be fp32 and have contiguous room for", M, N);
  Op e;
  if (given(p[7])) {
    e.epilogue = CUTHIP_EPI_UNARY;
    e.op = lookup(g_unary, p[7]);
  } else if (given(p[8])) {
    const char *bad = "matmul_sep: binary epilogue needs an fp32 D with the shape and stride of C";
    if (!given(p[9])) fail(bad);
    const at::Tensor &d = tensor(p[9]);
    if (d.sizes() != out.sizes() || d.scalar_type() != at::kFloat || d.stride(0) != out.stride(0) || !holds(d, M, N)) fail(bad);
    e.epilogue = CUTHIP_EPI_BINARY;
    e.op = lookup(g_binary, p[8]);
    e.d = ptr(d);
  }
  const int variant = (int)integer(p[10]);
  const size_t bytes = cuthip_matmul_sep_workspace_bytes_for(q4 ? CUTHIP_OP_MATMUL_Q4 : CUTHIP_OP_MATMUL_Q8, variant, (uint32_t)M, (uint32_t)K, (uint32_t)N);
  const at::Tensor ws = empty({(int64_t)std::max<size_t>(bytes, 1)}, at::kByte, in);
  const uint32_t sa = (uint32_t)a.stride(0), sb = (uint32_t)b.stride(0), sc = (uint32_t)out.stride(0), ss = (uint32_t)s.stride(0);
  if (q4)
    call(cuthip_matmul_q4_sep, (const float *)ptr(a), (const uint8_t *)ptr(b), (const uint16_t *)ptr(s), (const float *)e.d, (float *)mut(out), (uint32_t)M,
                               (uint32_t)K, (uint32_t)N, sa, sb, sc, ss, e.epilogue, e.op, affine, variant, mut(ws), bytes, stream());
  else
    call(cuthip_matmul_q8_sep, (const float *)ptr(a), (const int8_t *)ptr(b), (const uint16_t *)ptr(s), (const float *)e.d, (float *)mut(out), (uint32_t)M,
                               (uint32_t)K, (uint32_t)N, sa, sb, sc, ss, e.epilogue, e.op, variant, mut(ws), bytes, stream());
  return given(p[6]) ? ref(p[6]) : THPVariable_Wrap(out);
}

PyObject *prepare_sep(PyObject *const *p) {   // w_blocks, fmt, N, K, stride_b, scale_stride
  const int f = format(p[1]);
  if (f != CUTHIP_Q8_0 && f != CUTHIP_Q4_0 && f != CUTHIP_Q4_K) fail("prepare_sep: only Q8_0, Q4_0 and Q4_K have a separated layout");
  const at::Tensor &w = tensor(p[0]);
  const int64_t N = integer(p[2]), K = integer(p[3]);
  const bool q4 = f != CUTHIP_Q8_0;
  const int64_t width = q4 ? N / 2 : N, sb = given(p[4]) ? integer(p[4]) : (width + 3) & ~(int64_t)3, ss = given(p[5]) ? integer(p[5]) : (N + 3) & ~(int64_t)3;
  const at::Tensor b = empty({K, sb}, q4 ? at::kByte : at::kChar, w), s = empty({(f == CUTHIP_Q4_K ? 2 : 1) * (K / 32), ss}, at::kHalf, w);
  {   // the kernel writes every column up to the width; the padding beyond it is zero
    const Released r;
    if (sb > width) b.slice(1, width).zero_();
    if (ss > N) s.slice(1, N).zero_();
  }
  call(cuthip_prepare_sep, f, ptr(w), (uint32_t)N, (uint32_t)K, mut(b), (uint32_t)sb, (uint16_t *)mut(s), (uint32_t)ss, stream());
  PyObject *pair = PyTuple_New(2);
  if (!pair) throw PyError{};
  PyTuple_SET_ITEM(pair, 0, THPVariable_Wrap(b));
  PyTuple_SET_ITEM(pair, 1, THPVariable_Wrap(s));
  return pair;
}

PyObject *setup(PyObject *const *p) {   // CutHipError, FORMATS, UNARY, BINARY, NormCarry, RopeAppend, ctypes
  g_error = ref(p[0]);
  g_formats = ref(p[1]);
  g_unary = ref(p[2]);
  g_binary = ref(p[3]);
  g_norm_carry = ref(p[4]);
  g_rope_append = ref(p[5]);
  g_ctypes = ref(p[6]);
  return ref(Py_None);
}

template <PyObject *(*F)(PyObject *const *), int ARGS> PyObject *entry(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != ARGS) {
    PyErr_Format(PyExc_TypeError, "expected %d arguments, got %zd", ARGS, n);
    return nullptr;
  }
  try {
    return F(args);
  } catch (const PyError &) {
    return nullptr;
  }
  END_HANDLE_TH_ERRORS
}

#define ENTRY(name, args) {#name, (PyCFunction)(void (*)(void))entry<name, args>, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {ENTRY(setup, 7),           ENTRY(dequantize, 6),   ENTRY(matmul_gguf, 13),      ENTRY(norm_carry, 6),
                         ENTRY(rope_append, 9),     ENTRY(matmul_gguf_carry, 10), ENTRY(matmul_gguf_pair, 12), ENTRY(rmsnorm, 5),
                         ENTRY(attn_decode, 11),    ENTRY(silu_mul, 2),     ENTRY(matmul_gguf_argmax, 11), ENTRY(embedding_rows, 6),
                         ENTRY(matmul_sep, 11),     ENTRY(prepare_sep, 6),  {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host_ops", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host_ops(void) { return PyModule_Create(&module); }
