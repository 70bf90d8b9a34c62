// The launches of a step, made from Python with as little between them as there can be: one call checks the operands, makes
// the outputs and starts the kernels. A step of a short prompt is a hundred launches whose kernels take 3 to 20 us each, and
// what the host does between two of them is then what bounds it: through ctypes, with the checks and the outputs made in
// Python, a launch cost 10 to 22 us on the host, 5 to 9 here (the launch itself 2.5, an output 0.8).
//
// Every function here serves the plain case of the function of the same name in ops/hip.py, whose arguments it takes in
// order, and answers None where anything is another way (a type, a stride, an alignment, a tensor that is not on a GPU) or
// the launcher refuses: that function then goes its own, general way, which also says what is wrong. Nothing has been
// launched by then: a launch that failed, and a refusal behind a launch of the same call, are raised as `_run` of ops/hip.py raises
// them (what has run may have written to its operands, and is not to run twice). Like all of ops/hip.py, calls go to the
// current device's current stream.
#include <Python.h>

#include <vector>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/empty_strided.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "entry_points.h"

namespace {

using at::Tensor;

constexpr int64_t DECODE_MAX_TOKENS = 65535, MAX_SPLITS = 1024, ROWS64_MAX_ROWS = 128, ROWS64_SLICE_K = 512, ROW_SKEW = 8,
                  GATED_SKEW_MIN_ROWS = 5;      // as the constants of these names (or MAX_DECODE_..., OPERAND_ROW_SKEW) in ops/hip.py

hipStream_t stream() { return c10::hip::getCurrentHIPStream().stream(); }

// The arguments of a call in order. `bad` once one is not what was asked for: the call then answers None.
struct Args {
  PyObject* const* at;
  Py_ssize_t left;
  bool bad = false;

  PyObject* next() {
    if (left <= 0) {
      bad = true;
      return Py_None;
    }
    --left;
    return *at++;
  }
  // a GPU tensor; or, where it may be, None (null)
  const Tensor* maybe() {
    PyObject* o = next();
    if (o == Py_None) return nullptr;
    if (!THPVariable_Check(o)) {
      bad = true;
      return nullptr;
    }
    const Tensor& t = THPVariable_Unpack(o);
    if (!t.is_cuda()) bad = true;
    return &t;
  }
  const Tensor* tensor() {
    const Tensor* t = maybe();
    if (!t) bad = true;
    return t;
  }
  int64_t integer() {
    const int64_t v = PyLong_AsLongLong(next());
    if (v == -1 && PyErr_Occurred()) {
      PyErr_Clear();
      bad = true;
    }
    return v;
  }
  int i32() {
    const int64_t v = integer();
    if (v != (int)v) bad = true;
    return (int)v;
  }
  float number() {
    const double v = PyFloat_AsDouble(next());
    if (v == -1.0 && PyErr_Occurred()) {
      PyErr_Clear();
      bad = true;
    }
    return (float)v;
  }
  bool done() { return !bad && left == 0; }
};

void* ptr(const Tensor* t) { return t ? t->data_ptr() : nullptr; }
template <class T> T* typed(const Tensor* t) { return t ? (T*)t->data_ptr() : nullptr; }
bool aligned(const Tensor& t, uintptr_t bytes = 16) { return !((uintptr_t)t.data_ptr() % bytes); }
bool is(const Tensor& t, at::ScalarType type) { return t.scalar_type() == type; }
bool bf16(const Tensor& t) { return is(t, at::kBFloat16); }
bool f32(const Tensor& t) { return is(t, at::kFloat); }
// the kernels' number for a storage type, or below zero
int code(const Tensor& t) { return f32(t) ? 0 : bf16(t) ? 1 : -1; }
bool fits(int64_t v) { return v >= 0 && v <= 0x7fffffff; }

bool vector(const Tensor& t, at::ScalarType type, int64_t n) { return is(t, type) && t.dim() == 1 && t.size(0) == n && t.is_contiguous(); }
bool matrix(const Tensor& t, int64_t rows, int64_t columns) { return t.dim() == 2 && t.size(0) == rows && t.size(1) == columns; }
// rows that lie apart in whole 16-byte pieces, dense and aligned
bool pieces(const Tensor& x) { return x.dim() == 2 && x.stride(1) == 1 && x.stride(0) % 8 == 0 && aligned(x); }

// Python's lock, let go of: memory may have to be waited for, and so may a full queue, another thread's product or the timing of a
// product's algorithms, while other threads have work in Python. (ctypes lets go of it for a launcher, torch for a new tensor.)
struct Unlocked {
  PyThreadState* state = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(state); }
};

Tensor make(const Tensor& like, at::IntArrayRef sizes, at::ScalarType type) {
  Unlocked unlocked;
  return at::empty(sizes, like.options().dtype(type));
}
// rows of n numbers `skew` apart from each other
Tensor make_rows(const Tensor& like, int64_t rows, int64_t n, int64_t skew) {
  Unlocked unlocked;
  return at::empty_strided({rows, n}, {n + skew, 1}, like.options());
}

// Whether a launcher has refused its operands, which it does before it launches anything. An error where it is more than that: a failed
// launch (or an earlier one's failure, found only now), or a refusal `behind` a launch of this call.
template <class F> bool refused(const char* name, const F& launch, bool behind = false) {
  const int rc = [&] {
    Unlocked unlocked;
    return launch();
  }();
  if (rc == TS_OK) return false;
  if (rc != TS_LAUNCH_FAILED && !behind) return true;
  PyObject* hip = PyImport_ImportModule("tinyserve_llm_amd.ops.hip");
  PyObject* none = hip ? PyObject_CallMethod(hip, "_run", "si", name, rc) : nullptr;      // (raises for every answer but TS_OK)
  Py_XDECREF(hip);
  Py_XDECREF(none);
  throw python_error();
}
#define TS_REFUSED(NAME, CALL, ...) refused(NAME, [&] { return CALL; }, ##__VA_ARGS__)

PyObject* wrap(const Tensor& t) { return THPVariable_Wrap(t); }
PyObject* none() { Py_RETURN_NONE; }

// No two elements of a cache share a place.
bool apart(const Tensor& c) {
  int64_t st[4], sz[4];
  for (int i = 0; i < 4; ++i) {
    int j = i;
    const int64_t a = c.stride(i), b = c.size(i);
    for (; j > 0 && (st[j - 1] > a || (st[j - 1] == a && sz[j - 1] > b)); --j) st[j] = st[j - 1], sz[j] = sz[j - 1];
    st[j] = a, sz[j] = b;
  }
  int64_t span = 1;
  for (int i = 0; i < 4; ++i)
    if (sz[i] > 1) {
      if (st[i] < span) return false;
      span = st[i] * sz[i];
    }
  return true;
}

// A layer's caches [pages, page size, heads, head size], as _check_cache and _check_cache_pair of ops/hip.py want them.
bool caches(const Tensor& k, const Tensor& v, at::ScalarType type, int64_t heads, int64_t dim, int64_t vdim) {
  if (k.dim() != 4 || v.dim() != 4 || !is(k, type) || !is(v, type)) return false;
  if (k.size(2) != heads || k.size(3) != dim || v.size(2) != heads || v.size(3) != vdim || v.size(0) != k.size(0) || v.size(1) != k.size(1)) return false;
  return apart(k) && apart(v) && k.stride(3) == 1 && ((k.stride(0) | k.stride(1) | k.stride(2)) * k.element_size()) % 16 == 0 && aligned(k);
}

// ---- norms and the residual stream ----

PyObject* rmsnorm(Args a) {      // x, weight, eps, residual, want_residual -> (norm, sum or None)
  const Tensor *x = a.tensor(), *w = a.tensor();
  const float eps = a.number();
  const Tensor* res = a.maybe();
  const bool want = a.i32();
  if (!a.done() || x->dim() != 2 || !x->is_contiguous() || code(*x) < 0 || code(*w) < 0 || !vector(*w, w->scalar_type(), x->size(1))) return none();
  if (res && !(matrix(*res, x->size(0), x->size(1)) && is(*res, x->scalar_type()) && res->is_contiguous())) return none();
  if (!fits(x->size(0)) || !fits(x->size(1))) return none();
  Tensor out = make(*x, x->sizes(), x->scalar_type()), sum;
  if (res && want) sum = make(*x, x->sizes(), x->scalar_type());
  if (TS_REFUSED("rmsnorm",
                 ts_rmsnorm(ptr(&out), sum.defined() ? ptr(&sum) : nullptr, ptr(x), ptr(res), ptr(w), nullptr, x->size(0), x->size(1), eps, code(*x), code(*w),
                            stream())))
    return none();
  PyObject* second = !want ? none() : wrap(res ? sum : *x);
  return Py_BuildValue("(NN)", wrap(out), second);
}

// A branch's rows in parts: a tuple (parts [count, n, width]) or (one, its factor, the other, its factor).
struct Parts {
  const float* p = nullptr;
  int64_t stride = 0;
  int count = 0, scaled = 0;
  float fa = 1.f, fb = 1.f;
};
bool in_parts(const Args& a) { return a.left > 0 && PyTuple_Check(*a.at); }
Parts row_parts(Args& a, int64_t n, int64_t width) {
  PyObject* tuple = a.next();
  std::vector<PyObject*> items;
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(tuple); ++i) items.push_back(PyTuple_GET_ITEM(tuple, i));
  Args in{items.data(), (Py_ssize_t)items.size()};
  const bool one = in.left == 1;
  const Tensor* p = in.tensor();
  Parts parts;
  if (one) {
    a.bad |= !in.done() || !f32(*p) || p->dim() != 3 || p->size(1) != n || p->size(2) != width || !p->is_contiguous() || !fits(p->size(0)) || p->size(0) < 1;
    if (!a.bad) parts = {typed<float>(p), n * width, (int)p->size(0)};
    return parts;
  }
  const float fa = in.number();
  const Tensor* second = in.tensor();
  const float fb = in.number();
  a.bad |= !in.done();
  for (const Tensor* t : {p, second}) a.bad = a.bad || !f32(*t) || !matrix(*t, n, width) || !t->is_contiguous();
  const int64_t apart = a.bad ? 0 : (char*)second->data_ptr() - (char*)p->data_ptr();
  a.bad |= apart % 4 != 0;
  if (!a.bad) parts = {typed<float>(p), apart / 4, 2, 1, fa, fb};
  return parts;
}

// A branch's rows as experts have left them: a tuple (rows, weights, shared, its gate, chosen experts, experts with matrices, input), as moe_combine of
// ops/hip.py takes them.
PyObject* post_norm_of_experts(const Tensor* x, Args& a) {
  PyObject* tuple = a.next();
  PyObject* items[7];
  for (int i = 0; i < 7; ++i) items[i] = PyTuple_GET_ITEM(tuple, i);
  Args in{items, 7};
  const Tensor *rows = in.tensor(), *weights = in.tensor(), *shared = in.maybe(), *gate = in.maybe(), *ids = in.maybe();
  const int real = in.i32();
  const Tensor* input = in.maybe();
  const Tensor *post = a.tensor(), *scale = a.maybe();
  const float post_eps = a.number();
  const Tensor* w = a.maybe();
  const float eps = a.number();
  const int out_code = a.i32();
  if (!in.done() || !a.done() || out_code < 0 || out_code > 1 || !f32(*x) || !x->is_contiguous() || weights->dim() != 2) return none();
  const int64_t n = x->size(0), width = x->size(1), top = weights->size(1);
  if (!f32(*weights) || weights->size(0) != n || !weights->is_contiguous() || top < 1 || !fits(n * top) || !fits(width)) return none();
  if (!f32(*rows) || !matrix(*rows, n * top, width) || !rows->is_contiguous()) return none();
  if (shared && !(f32(*shared) && matrix(*shared, n, width) && shared->is_contiguous())) return none();
  if (gate && !(shared && f32(*gate) && gate->numel() == n && gate->is_contiguous())) return none();
  if (ids && !(input && is(*ids, at::kInt) && matrix(*ids, n, top) && ids->is_contiguous() && bf16(*input) && matrix(*input, n, width) && input->is_contiguous())) return none();
  for (const Tensor* v : {post, scale, w})
    if (v && !vector(*v, at::kFloat, width)) return none();
  Tensor out = make(*x, {n, width}, out_code ? at::kBFloat16 : at::kFloat);
  if (TS_REFUSED("stream_post_norm",
                 ts_stream_post_norm_experts(typed<float>(x), typed<float>(rows), typed<float>(weights), typed<float>(shared), top, typed<int32_t>(ids), real, ptr(input),
                                             typed<float>(gate), typed<float>(post), typed<float>(scale), post_eps, ptr(&out), out_code, typed<float>(w), eps, n, width,
                                             stream())))
    return none();
  return wrap(out);
}

PyObject* stream_post_norm(Args a) {      // x, a (or in parts, or as experts left it), post weight, scale, post eps, weight, eps, out code or -1 -> rows or None
  const Tensor* x = a.tensor();
  if (in_parts(a)) {
    if (a.bad || x->dim() != 2) return none();
    if (PyTuple_GET_SIZE(*a.at) == 7) return post_norm_of_experts(x, a);
    const int64_t n = x->size(0), width = x->size(1);
    const Parts b = row_parts(a, n, width);
    const Tensor *post = a.tensor(), *scale = a.maybe();
    const float post_eps = a.number();
    const Tensor* w = a.maybe();
    const float eps = a.number();
    const int out_code = a.i32();
    if (!a.done() || out_code < 0 || out_code > 1 || !f32(*x) || !x->is_contiguous() || !fits(n) || !fits(width)) return none();
    for (const Tensor* v : {post, scale, w})
      if (v && !vector(*v, at::kFloat, width)) return none();
    Tensor out = make(*x, {n, width}, out_code ? at::kBFloat16 : at::kFloat);
    if (TS_REFUSED("stream_post_norm",
                   ts_stream_post_norm_parts(typed<float>(x), b.p, b.stride, b.count, b.scaled, b.fa, b.fb, typed<float>(post), typed<float>(scale), post_eps, ptr(&out),
                                             out_code, typed<float>(w), eps, n, width, stream())))
      return none();
    return wrap(out);
  }
  const Tensor *b = a.tensor(), *post = a.tensor(), *scale = a.maybe();
  const float post_eps = a.number();
  const Tensor* w = a.maybe();
  const float eps = a.number();
  const int out_code = a.i32();
  if (!a.done() || out_code < 0 || out_code > 1 || !f32(*x) || x->dim() != 2 || !x->is_contiguous()) return none();
  const int64_t n = x->size(0), width = x->size(1);
  if (!f32(*b) || !matrix(*b, n, width) || !b->is_contiguous() || !fits(n) || !fits(width)) return none();
  for (const Tensor* v : {post, scale, w})
    if (v && !vector(*v, at::kFloat, width)) return none();
  Tensor out = make(*x, {n, width}, out_code ? at::kBFloat16 : at::kFloat);
  if (TS_REFUSED("stream_post_norm",
                 ts_stream_post_norm(typed<float>(x), typed<float>(b), typed<float>(post), typed<float>(scale), post_eps, ptr(&out), out_code, typed<float>(w),
                                     eps, n, width, stream())))
    return none();
  return wrap(out);
}

PyObject* stream_update_norm(Args a) {      // x, a, b (or in parts), mult, weight, eps, out code -> rows (one norm, no bias, no picked rows)
  const Tensor *x = a.tensor(), *b1 = a.maybe();
  if (in_parts(a)) {
    if (a.bad || x->dim() != 2) return none();
    const int64_t n = x->size(0), width = x->size(1);
    const Parts b = row_parts(a, n, width);
    const float mult = a.number();
    const Tensor* w = a.tensor();
    const float eps = a.number();
    const int out_code = a.i32();
    if (!a.done() || out_code < 0 || out_code > 1 || !f32(*x) || !x->is_contiguous() || code(*w) < 0 || !vector(*w, w->scalar_type(), width)) return none();
    if ((b1 && !(f32(*b1) && matrix(*b1, n, width) && b1->is_contiguous())) || !fits(n) || !fits(width)) return none();
    Tensor out = make(*x, {n, width}, out_code ? at::kBFloat16 : at::kFloat);
    if (TS_REFUSED("stream_update_norm",
                   ts_stream_update_norm_parts(typed<float>(x), typed<float>(b1), b.p, b.stride, b.count, b.scaled, b.fa, b.fb, mult, ptr(&out), out_code, ptr(w),
                                               code(*w), eps, n, width, stream())))
      return none();
    return wrap(out);
  }
  const Tensor* b2 = a.maybe();
  const float mult = a.number();
  const Tensor* w = a.tensor();
  const float eps = a.number();
  const int out_code = a.i32();
  if (!a.done() || out_code < 0 || out_code > 1 || !f32(*x) || x->dim() != 2 || !x->is_contiguous()) return none();
  const int64_t n = x->size(0), width = x->size(1);
  for (const Tensor* t : {b1, b2})
    if (t && !(matrix(*t, n, width) && t->is_contiguous() && code(*t) >= 0)) return none();
  if (code(*w) < 0 || !vector(*w, w->scalar_type(), width) || !fits(n) || !fits(width)) return none();
  Tensor out = make(*x, {n, width}, out_code ? at::kBFloat16 : at::kFloat);
  if (TS_REFUSED("stream_update_norm",
                 ts_stream_update_norm(typed<float>(x), ptr(b1), b1 ? code(*b1) : 0, ptr(b2), b2 ? code(*b2) : 0, nullptr, 0, mult, ptr(&out), nullptr,
                                       out_code, ptr(w), nullptr, code(*w), eps, nullptr, n, width, stream())))
    return none();
  return wrap(out);
}

// ---- products ----

PyObject* gemm_library(Args a) {      // x, weight, 32-bit out -> y
  const Tensor *x = a.tensor(), *w = a.tensor();
  const bool wide = a.i32();
  if (!a.done() || x->dim() != 2 || w->dim() != 2 || !bf16(*x) || !bf16(*w) || x->size(1) != w->size(1) || x->stride(1) != 1 || w->stride(1) != 1) return none();
  const int64_t M = x->size(0), K = x->size(1), N = w->size(0);
  if (!M || !N || !fits(M) || !fits(N) || !fits(K)) return none();
  Tensor y = make(*x, {M, N}, wide ? at::kFloat : at::kBFloat16);
  if (TS_REFUSED("gemm_library",
                 ts_gemm_library_bf16(ptr(&y), ptr(x), ptr(w), M, N, K, x->stride(0), w->stride(0), N, wide, 0, nullptr, 0, stream())))
    return none();
  return wrap(y);
}

bool packed16(const Tensor& p, int64_t K) {
  return bf16(p) && p.dim() == 4 && p.size(1) * 32 == K && p.size(2) == 64 && p.size(3) == 8 && p.is_contiguous();
}

// The products of a group (`gemm_group` of ops/hip.py), 32 bits on their way out: by the kernel that streams W past x where `packed` is given (the copies
// of all the weights one behind the other), else in whole tiles (`tile`: and from its bit 8 on a bit for each product in chains).
PyObject* group(PyObject* xs, PyObject* ws, const Tensor* packed, int tile) {
  constexpr Py_ssize_t most{8};
  if (!PyTuple_Check(xs) || !PyTuple_Check(ws)) return none();
  const Py_ssize_t n = PyTuple_GET_SIZE(xs);
  if (n < 1 || n > most || PyTuple_GET_SIZE(ws) != n) return none();
  const Tensor *x[most], *w[most];
  const void *xp[most], *wp[most];
  void* yp[most];
  int widths[most];
  int64_t N = 0;
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject *px = PyTuple_GET_ITEM(xs, i), *pw = PyTuple_GET_ITEM(ws, i);
    if (!THPVariable_Check(px) || !THPVariable_Check(pw)) return none();
    x[i] = &THPVariable_Unpack(px), w[i] = &THPVariable_Unpack(pw);
    if (!x[i]->is_cuda() || !w[i]->is_cuda() || w[i]->dim() != 2 || !bf16(*x[i]) || !bf16(*w[i]) || !pieces(*x[i]) || !pieces(*w[i])) return none();
    if (x[i]->sizes() != x[0]->sizes() || x[i]->strides() != x[0]->strides() || w[i]->strides() != w[0]->strides()) return none();
    if (w[i]->size(1) != x[0]->size(1) || w[i]->size(0) < 8 || w[i]->size(0) % 8 || !fits(w[i]->size(0))) return none();
    widths[i] = w[i]->size(0), xp[i] = ptr(x[i]), wp[i] = ptr(w[i]), N += widths[i];
  }
  const int64_t M = x[0]->size(0), K = x[0]->size(1), ldx = x[0]->stride(0), ldw = w[0]->stride(0);
  if (M < 1 || !fits(M) || !fits(K) || K % 64 || K < 192 || ldx < K || ldw < K || 512 * ldx >= 1LL << 31 || 512 * ldw >= 1LL << 31) return none();
  if (packed) {
    if (!packed16(*packed, K) || packed->size(0) * 16 != N || M > ROWS64_MAX_ROWS || K % 1024) return none();
    for (Py_ssize_t i = 0; i < n; ++i)
      if (widths[i] % 16) return none();
  }
  Tensor y[most];
  for (Py_ssize_t i = 0; i < n; ++i) y[i] = make(*x[0], {M, widths[i]}, at::kFloat), yp[i] = ptr(&y[i]);
  if (packed ? TS_REFUSED("gemm_rows64_group", ts_gemm_rows64_group_bf16(n, yp, xp, ptr(packed), widths, M, K, ldx, stream()))
             : TS_REFUSED("gemm_whole", ts_gemm_whole_bf16(n, yp, xp, wp, widths, M, K, ldx, ldw, tile & 0xff, tile >> 8, 1, stream())))
    return none();
  PyObject* out = PyTuple_New(n);
  for (Py_ssize_t i = 0; out && i < n; ++i) PyTuple_SET_ITEM(out, i, wrap(y[i]));
  return out;
}

// x, weight, tile, slices, 32-bit out, residual, norm weight, eps -> y, or with a norm weight (norm, sum); x, weight, tile, slices, 32-bit out -> the slices'
// parts; or, with tuples of operands: operands,
// weights, tile, packed copies -> the products of a `group`
PyObject* gemm_slices(Args a) {
  if (a.left == 4) {
    PyObject *xs = a.next(), *ws = a.next();
    const int tile = a.i32();
    const Tensor* packed = a.maybe();
    return a.done() ? group(xs, ws, packed, tile) : none();
  }
  const bool leave = a.left == 5;
  const Tensor *x = a.tensor(), *w = a.tensor();
  const int tile = a.i32(), slices = a.i32();
  const bool wide = a.i32();
  const Tensor *res = leave ? nullptr : a.maybe(), *nw = leave ? nullptr : a.maybe();
  const float eps = leave ? 0.f : a.number();
  if (!a.done() || x->dim() != 2 || w->dim() != 2 || !bf16(*x) || !bf16(*w) || x->size(1) != w->size(1) || !pieces(*x) || !pieces(*w)) return none();
  const int64_t M = x->size(0), K = x->size(1), N = w->size(0);
  if (!M || !N || !fits(M) || !fits(N) || !fits(K) || x->stride(0) < K || w->stride(0) < K || slices < 1 || slices > 64 || (res && !nw)) return none();
  if (nw && (wide || !vector(*nw, at::kBFloat16, N) || !aligned(*nw))) return none();
  if (res && !(bf16(*res) && matrix(*res, M, N) && res->is_contiguous() && aligned(*res))) return none();
  if (N % 8 || K % 64) return none();
  if (leave) {
    if (!wide) return none();
    Tensor parts = make(*x, {slices, M, N}, at::kFloat);
    if (TS_REFUSED("gemm_slices", ts_gemm_slices_parts_bf16(typed<float>(&parts), ptr(x), ptr(w), M, N, K, x->stride(0), w->stride(0), tile, slices, stream()))) return none();
    return wrap(parts);
  }
  Tensor parts, y = make(*x, {M, N}, wide ? at::kFloat : at::kBFloat16), sum;
  if (nw || slices > 1) parts = make(*x, {slices, M, N}, at::kFloat);
  if (nw) sum = make(*x, {M, N}, at::kBFloat16);
  if (TS_REFUSED("gemm_slices",
                 ts_gemm_slices_bf16(ptr(&y), nw ? ptr(&sum) : nullptr, parts.defined() ? ptr(&parts) : nullptr, ptr(x), ptr(w), M, N, K, x->stride(0), w->stride(0), tile, slices, wide,
                                     ptr(res), ptr(nw), eps, stream())))
    return none();
  return nw ? Py_BuildValue("(NN)", wrap(y), wrap(sum)) : wrap(y);
}

PyObject* gemm_glu(Args a) {      // x, weight, tile, form's number, limit, slope, up_shift -> y
  const Tensor *x = a.tensor(), *w = a.tensor();
  const int tile = a.i32(), form = a.i32();
  const float limit = a.number(), slope = a.number(), shift = a.number();
  if (!a.done() || x->dim() != 2 || w->dim() != 2 || !bf16(*x) || !bf16(*w) || x->size(1) != w->size(1) || !pieces(*x) || !pieces(*w)) return none();
  const int64_t M = x->size(0), K = x->size(1), F = w->size(0) / 2;
  if (!M || !F || !fits(M) || !fits(w->size(0)) || w->size(0) % 16 || K % 64 || x->stride(0) < K || w->stride(0) < K) return none();
  Tensor y = make(*x, {M, F}, at::kBFloat16);
  if (TS_REFUSED("gemm_glu",
                 ts_gemm_glu_bf16(ptr(&y), ptr(x), ptr(w), M, F, K, x->stride(0), w->stride(0), F, tile, form, limit, slope, shift, stream())))
    return none();
  return wrap(y);
}

bool squares_fit(const Tensor* s, int64_t rows) { return !s || (f32(*s) && s->dim() == 2 && s->size(0) == rows && s->size(1) >= 1 && s->is_contiguous()); }

// What gemm_rows64 makes of up to 8 rows of x and the copy that the 8-row form reads (five-dimensional: hip.pack_weight8).
PyObject* rows8(const Tensor& x, const Tensor& p, bool wide, float cap) {
  const int64_t M = x.size(0), K = x.size(1), N = p.size(0) * 8;
  if (M < 1 || M > 8 || !fits(N) || !fits(K) || !bf16(p) || p.size(2) != ts_skinny8_steps(K) || p.size(1) * p.size(2) * 64 != K || p.size(3) != 64 || p.size(4) != 8 ||
      !p.is_contiguous())
    return none();
  Tensor y = make(x, {M, N}, wide ? at::kFloat : at::kBFloat16);
  if (TS_REFUSED("gemm_skinny8", ts_gemm_skinny8_bf16(ptr(&y), ptr(&x), ptr(&p), M, N, K, x.stride(0), K, N, wide ? 0 : 1, 1, nullptr, nullptr, nullptr, nullptr, nullptr,
                                                      0, nullptr, nullptr, nullptr, 0, 0, 0, 0, cap, stream())))
    return none();
  return wrap(y);
}

PyObject* gemm_rows64(Args a) {      // x, packed, 32-bit out, unit's number (0: none), squares, eps, limit (0: none; without a unit the sums' cap), slope, up_shift, `few` of the launcher if it is there -> y
  const Tensor *x = a.tensor(), *p = a.tensor();
  const bool wide = a.i32();
  const int unit = a.i32();
  const Tensor* sq = a.maybe();
  const float eps = a.number(), limit = a.number(), slope = a.number(), shift = a.number();
  const int few = a.left ? a.i32() : 0, steps = few > 1 ? few : 0;
  if (a.done() && p->dim() == 5) return unit || sq || few || x->dim() != 2 || !bf16(*x) || !pieces(*x) ? none() : rows8(*x, *p, wide, limit);
  if (!a.done() || x->dim() != 2 || !bf16(*x) || !pieces(*x) || !packed16(*p, x->size(1)) || (unit && wide) || (unit > 1 && sq)) return none();
  const int64_t M = x->size(0), K = x->size(1), N = p->size(0) * 16;
  if (M < 1 || M > ROWS64_MAX_ROWS || N % (unit ? 128 : 64) || K % 1024 || !squares_fit(sq, M) || !fits(N) || !fits(K)) return none();
  if (steps && (!unit || M > 8 || (steps != 4 && steps != 8 && steps != 16) || N / 2 % (64 * steps))) return none();
  const int64_t skew = M >= GATED_SKEW_MIN_ROWS ? ROW_SKEW : 0;
  Tensor y = steps  ? make(*x, {N / 2 / (64 * steps), steps, 64, 8}, at::kBFloat16)
             : unit ? make_rows(*x, M, N / 2, skew)
                    : make(*x, {M, N}, wide ? at::kFloat : at::kBFloat16);
  if (TS_REFUSED("gemm_rows64",
                 ts_gemm_rows64_bf16(ptr(&y), ptr(x), ptr(p), M, N, K, x->stride(0), steps ? N / 2 : y.stride(0), unit, wide, ptr(sq), sq ? sq->size(1) : 0,
                                     eps, limit, slope, shift, few, stream())))
    return none();
  return wrap(y);
}

PyObject* gemm_rows64_sliced(Args a) {      // x, packed, slices (0: whole, by the kernel that streams the copy; with a weight), residual, norm weight -> y, or with a weight (sum, operand, squares)
  const Tensor *x = a.tensor(), *p = a.tensor();
  const int slices = a.i32();
  const Tensor *res = a.maybe(), *nw = a.maybe();
  if (!a.done() || x->dim() != 2 || !bf16(*x) || !pieces(*x) || !packed16(*p, x->size(1)) || (res && !nw)) return none();
  const int64_t M = x->size(0), K = x->size(1), N = p->size(0) * 16;
  if (M < 1 || M > ROWS64_MAX_ROWS || !fits(N) || !fits(K) || (!slices && !nw)) return none();
  if (slices && (N % 64 || slices < 1 || slices > 64 || K % (ROWS64_SLICE_K * slices))) return none();
  if (nw && !vector(*nw, at::kBFloat16, N)) return none();
  if (res && !(bf16(*res) && matrix(*res, M, N) && res->is_contiguous())) return none();
  if (!slices) {
    if (x->stride(0) < K || !aligned(*p)) return none();
    const int64_t tiles = [&] {
      Unlocked unlocked;
      return ts_skinny_tiles(M, N, K);
    }();
    Tensor sum = make(*x, {M, N}, at::kBFloat16), operand = make(*x, {M, N}, at::kBFloat16), squares = make(*x, {M, tiles}, at::kFloat);
    if (TS_REFUSED("gemm_skinny", ts_gemm_skinny_bf16(nullptr, ptr(x), ptr(p), nullptr, nullptr, nullptr, M, N, K, x->stride(0), K, N, 0.f, 0, 0, 1, 1, nullptr, 0,
                                                      ptr(res), ptr(nw), ptr(&sum), ptr(&operand), ptr(&squares), 0, 0.f, 0.f, 0.f, stream())))
      return none();
    return Py_BuildValue("(NNN)", wrap(sum), wrap(operand), wrap(squares));
  }
  Tensor parts = make(*x, {slices, M, N}, at::kFloat);
  if (!nw) {
    Tensor y = make(*x, {M, N}, at::kBFloat16);
    if (TS_REFUSED("gemm_rows64_sliced",
                   ts_gemm_rows64_sliced_bf16(ptr(&y), ptr(&parts), ptr(x), ptr(p), M, N, K, x->stride(0), slices, nullptr, nullptr, nullptr, nullptr, nullptr,
                                              0, stream())))
      return none();
    return wrap(y);
  }
  Tensor sum = make(*x, {M, N}, at::kBFloat16), operand = make_rows(*x, M, N, ROW_SKEW), squares = make(*x, {M, 1}, at::kFloat);
  if (TS_REFUSED("gemm_rows64_sliced",
                 ts_gemm_rows64_sliced_bf16(nullptr, ptr(&parts), ptr(x), ptr(p), M, N, K, x->stride(0), slices, ptr(res), ptr(nw), ptr(&sum), ptr(&operand),
                                            ptr(&squares), operand.stride(0), stream())))
    return none();
  return Py_BuildValue("(NNN)", wrap(sum), wrap(operand), wrap(squares));
}

// ---- projections on their way into the cache ----

struct Store {      // where keys and values go; without caches nothing is written
  const Tensor *slots, *k, *v;
  int64_t page = 1, ks[3] = {0, 0, 0}, vs[4] = {0, 0, 0, 0};

  bool take(int64_t rows, at::ScalarType type, int64_t heads, int64_t dim, int64_t vdim) {
    if (!k) return true;
    if (!v || !slots || !vector(*slots, at::kInt, rows) || !caches(*k, *v, type, heads, dim, vdim)) return false;
    page = k->size(1);
    for (int i = 0; i < 3; ++i) ks[i] = k->stride(i);
    for (int i = 0; i < 4; ++i) vs[i] = v->stride(i);
    return true;
  }
};

PyObject* rope_store(Args a) {      // qkv, table, positions, slots, k, v, heads, kv heads, head size -> q
  const Tensor *x = a.tensor(), *table = a.maybe(), *pos = a.tensor();
  Store s{a.maybe(), a.maybe(), a.maybe()};
  const int nh = a.i32(), nkv = a.i32(), hd = a.i32();
  if (!a.done() || x->dim() != 2 || code(*x) < 0 || !x->is_contiguous() || nh <= 0 || nkv < 0 || hd <= 0) return none();
  const int64_t T = x->size(0);
  if (x->size(1) != (nh + 2 * (int64_t)nkv) * hd || !vector(*pos, at::kInt, T) || !fits(T)) return none();
  if (table && !(f32(*table) && table->dim() == 2 && table->is_contiguous() && table->size(1) >= 2 && table->size(1) <= hd && table->size(1) % 2 == 0)) return none();
  if (!s.take(T, x->scalar_type(), nkv, hd, hd)) return none();
  Tensor q = make(*x, {T, nh, hd}, x->scalar_type());
  if (TS_REFUSED("rope_store",
                 ts_rope_store(ptr(&q), ptr(s.k), ptr(s.v), ptr(x), typed<float>(table), typed<int32_t>(pos), typed<int32_t>(s.slots), T, nh, nkv, hd, table ?
                               table->size(1) : hd, table != nullptr, s.page, s.ks[0], s.ks[1], s.ks[2], s.vs[0], s.vs[1], s.vs[2], s.vs[3], code(*x),
                               stream())))
    return none();
  return wrap(q);
}

// x, packed, slices, table, positions, slots, k, v, heads, kv heads, head size, eps, squares -> q; or, for `qkv_rope_store_whole`, the weight as it is
// in the packed one's place and the tile in the slices'
PyObject* qkv_rope_store_sliced(Args a) {
  const Tensor *x = a.tensor(), *p = a.tensor();
  const int slices = a.i32();
  const Tensor *table = a.maybe(), *pos = a.tensor();
  Store s{a.maybe(), a.maybe(), a.maybe()};
  const int nh = a.i32(), nkv = a.i32(), hd = a.i32();
  const float eps = a.number();
  const Tensor* sq = a.maybe();
  if (!a.done() || x->dim() != 2 || !bf16(*x) || !pieces(*x) || nh <= 0 || nkv < 0 || hd <= 0 || hd % 32) return none();
  const int64_t M = x->size(0), K = x->size(1);
  if (p->dim() == 2) {
    const int64_t N = (nh + 2 * (int64_t)nkv) * hd;
    if (!bf16(*p) || !pieces(*p) || !matrix(*p, N, K) || sq || !M || !fits(M) || !fits(N) || !fits(K) || x->stride(0) < K || p->stride(0) < K) return none();
    if (!vector(*pos, at::kInt, M) || !s.take(M, at::kBFloat16, nkv, hd, hd)) return none();
    if (table && !(f32(*table) && table->dim() == 2 && table->size(1) == hd && table->is_contiguous())) return none();
    Tensor q = make(*x, {M, nh, hd}, at::kBFloat16);
    if (TS_REFUSED("qkv_rope_store_whole",
                   ts_gemm_whole_rope_bf16(ptr(&q), ptr(x), ptr(p), M, K, x->stride(0), p->stride(0), typed<float>(table), typed<int32_t>(pos), typed<int32_t>(s.slots),
                                           ptr(s.k), ptr(s.v), nh, nkv, hd, s.page, s.ks[0], s.ks[1], s.ks[2], s.vs[0], s.vs[1], s.vs[2], s.vs[3], slices, stream())))
      return none();
    return wrap(q);
  }
  if (!packed16(*p, K) || !aligned(*p)) return none();
  const int64_t N = p->size(0) * 16;
  if (N != (nh + 2 * (int64_t)nkv) * hd || M < 1 || M > ROWS64_MAX_ROWS) return none();
  if (slices && (N % 64 || slices < 1 || slices > 64 || K % (ROWS64_SLICE_K * slices))) return none();
  if (!vector(*pos, at::kInt, M) || !squares_fit(sq, M) || !fits(N) || !fits(K)) return none();
  if (table && !(f32(*table) && table->dim() == 2 && table->size(1) == hd && table->is_contiguous())) return none();
  if (!s.take(M, at::kBFloat16, nkv, hd, hd)) return none();
  Tensor q = make(*x, {M, nh, hd}, at::kBFloat16);
  if (!slices) {      // whole, by the kernel that streams the copy
    if (TS_REFUSED("qkv_rope_store",
                   ts_gemm_skinny_rope_bf16(ptr(&q), ptr(x), ptr(p), nullptr, nullptr, nullptr, M, K, x->stride(0), K, eps, sq ? 2 : 0, 1, typed<float>(table),
                                            typed<int32_t>(pos), typed<int32_t>(s.slots), ptr(s.k), ptr(s.v), nh, nkv, hd, table != nullptr, s.page, s.ks[0],
                                            s.ks[1], s.ks[2], s.vs[0], s.vs[1], s.vs[2], s.vs[3], ptr(sq), sq ? sq->size(1) : 0, stream())))
      return none();
    return wrap(q);
  }
  Tensor parts = make(*x, {slices, M, N}, at::kFloat);
  if (TS_REFUSED("qkv_rope_store_sliced",
                 ts_gemm_rows64_sliced_rope_bf16(ptr(&q), ptr(&parts), ptr(x), ptr(p), M, K, x->stride(0), slices, ptr(sq), sq ? sq->size(1) : 0, eps,
                                                 typed<float>(table), typed<int32_t>(pos), typed<int32_t>(s.slots), ptr(s.k), ptr(s.v), nh, nkv, hd, table !=
                                                 nullptr, s.page, s.ks[0], s.ks[1], s.ks[2], s.vs[0], s.vs[1], s.vs[2], s.vs[3], stream())))
    return none();
  return wrap(q);
}

PyObject* qkv_finish(Args a) {      // qkv, freqs, positions, slots, k, v, heads, kv heads, head size, value size, out code, interleaved, qk eps or None, v eps or None, amplitude -> q
  const Tensor *x = a.tensor(), *freqs = a.maybe(), *pos = a.tensor();
  Store s{a.maybe(), a.maybe(), a.maybe()};
  const int nh = a.i32(), nkv = a.i32(), hd = a.i32(), vd = a.i32(), out_code = a.i32(), interleaved = a.i32();
  float eps[2];
  int normed[2];
  for (int i = 0; i < 2; ++i) {
    normed[i] = a.left > 0 && *a.at != Py_None;
    eps[i] = normed[i] ? a.number() : (a.next(), 0.f);
  }
  const float amplitude = a.number();
  if (!a.done() || out_code < 0 || out_code > 1 || x->dim() != 2 || !x->is_contiguous() || nh <= 0 || nkv < 0 || hd <= 0 || hd > 256 || vd <= 0 || vd > 256) return none();
  const at::ScalarType out_type = out_code ? at::kBFloat16 : at::kFloat;
  const int64_t T = x->size(0);
  if (x->size(1) < (nh + (int64_t)nkv) * hd + (int64_t)nkv * vd || !(f32(*x) || is(*x, out_type)) || !vector(*pos, at::kInt, T) || !fits(T)) return none();
  if (freqs && !(is(*freqs, at::kDouble) && freqs->dim() == 1 && freqs->is_contiguous() && 2 * freqs->size(0) <= hd)) return none();
  if (!s.take(T, out_type, nkv, hd, vd)) return none();
  Tensor q = make(*x, {T, nh, hd}, out_type);
  if (TS_REFUSED("qkv_finish",
                 ts_qkv_finish(ptr(&q), ptr(s.k), ptr(s.v), ptr(x), typed<double>(freqs), typed<int32_t>(pos), typed<int32_t>(s.slots), T, nh, nkv, hd, vd,
                               freqs ? 2 * freqs->size(0) : 0, interleaved, normed[0], eps[0], normed[1], eps[1], s.page, s.ks[0], s.ks[1], s.ks[2], s.vs[0],
                               s.vs[1], s.vs[2], s.vs[3], code(*x), out_code, amplitude, x->size(1), stream())))
    return none();
  return wrap(q);
}

// ---- attention ----

// The stride between a gate's rows as the kernels take it: below zero for a number per head. False: no gate of this attention.
bool gate_stride(const Tensor* g, int64_t rows, int64_t heads, int64_t dim, int64_t* stride) {
  *stride = 0;
  if (!g) return true;
  if (!f32(*g) || g->dim() != 2 || g->size(0) != rows || g->stride(1) != 1) return false;
  const bool per_head = g->size(1) == heads && dim != 1;
  if (!(per_head || g->size(1) == heads * dim) || g->stride(0) < g->size(1)) return false;
  *stride = per_head ? -g->stride(0) : g->stride(0);
  return true;
}

// A step with portions of prompts: the first `lead` tokens, one a request, by the split-key kernel, the others by the kernel that
// takes tiles of tokens. q, k, v, block tables, request of token, positions, tiles, scale, window, softcap, sink, sinks, slopes,
// gate, table pages an entry, lead, keys and waves a workgroup of the split walk, tokens a tile, waves, chunks, keys a chunk, first
// token of the tiles -> out [tokens, heads, head size]
PyObject* attention_step(Args a) {
  const Tensor *q = a.tensor(), *k = a.tensor(), *v = a.tensor(), *tables = a.tensor(), *seq = a.tensor(), *pos = a.tensor(), *tiles = a.tensor();
  const float scale = a.number();
  const int window = a.i32();
  const float softcap = a.number();
  const int sink = a.i32();
  const Tensor *sinks = a.maybe(), *slopes = a.maybe(), *gate = a.maybe();
  const int64_t per_entry = a.integer(), lead = a.integer();
  const int dchunk = a.i32(), dwaves = a.i32(), tile_tokens = a.i32(), waves = a.i32(), splits = a.i32(), chunk = a.i32();
  const int64_t first = a.integer();
  if (!a.done() || q->dim() != 3 || !q->is_contiguous() || !bf16(*q) || k->dim() != 4) return none();
  const int64_t T = q->size(0), nh = q->size(1), hd = q->size(2), page = k->size(1), nkv = k->size(2);
  if (!nkv || nh % nkv || !caches(*k, *v, at::kBFloat16, nkv, hd, hd) || !fits(T)) return none();
  const int64_t group = nh / nkv;
  if (!(hd == 32 || hd == 64 || hd == 96 || hd == 128) || group > 16 || group * hd > 2048 || page % 8 || v->stride(1) != 1 || !aligned(*v)) return none();
  if ((k->stride(0) | k->stride(1) | k->stride(2) | v->stride(0) | v->stride(2) | v->stride(3)) % 8) return none();
  if (!is(*tables, at::kInt) || tables->dim() != 2 || !tables->is_contiguous() || !vector(*seq, at::kInt, T) || !vector(*pos, at::kInt, T)) return none();
  if (!is(*tiles, at::kInt) || tiles->dim() != 2 || tiles->size(1) != 2 || !tiles->is_contiguous()) return none();
  for (const Tensor* t : {sinks, slopes})
    if (t && !vector(*t, at::kFloat, nh)) return none();
  int64_t gstride;
  const bool general = softcap > 0 || sink || sinks || slopes || gate;
  if (!gate_stride(gate, T, nh, hd, &gstride) || (general && page % 32)) return none();
  if (per_entry < 1 || per_entry > 65536 || (per_entry & (per_entry - 1)) || lead < 0 || lead >= T || lead > DECODE_MAX_TOKENS) return none();
  const int run = __builtin_ctzll(per_entry);
  const bool two = waves == 8 && (hd == 64 || hd == 128);
  const int64_t per_wave = waves * (16 / group);
  if (!(waves == 4 || two) || !(tile_tokens == per_wave || tile_tokens == 2 * per_wave || (tile_tokens == 4 * per_wave && waves == 4))) return none();
  if (splits < 1 || splits > MAX_SPLITS || (splits > 1 && (chunk <= 0 || chunk % 32)) || first < 0 || first >= T) return none();
  const int64_t blocks = tables->size(1), capacity = blocks * per_entry * page;
  int64_t dsplits = 1;
  if (lead) {
    const int most = hd > 64 && dchunk != 32 * dwaves ? 4 : 8;
    if (dwaves < 1 || dwaves > most || dchunk <= 0 || dchunk % (32 * dwaves) || 4 * (32 * dwaves + dwaves * group * hd) > 65536) return none();
    dsplits = (capacity + dchunk - 1) / dchunk;
    if (dsplits > MAX_SPLITS) return none();
  }
  Tensor out = make(*q, q->sizes(), at::kBFloat16), po, pm, dpo, dpm;
  if (splits > 1) po = make(*q, {T, nh, splits, hd}, at::kFloat), pm = make(*q, {T, nh, splits, 2}, at::kFloat);
  if (dsplits > 1) dpo = make(*q, {lead, nh, dsplits, hd}, at::kFloat), dpm = make(*q, {lead, nh, dsplits, 2}, at::kFloat);
  float *pof = splits > 1 ? typed<float>(&po) : nullptr, *pmf = splits > 1 ? typed<float>(&pm) : nullptr;
  float *dpof = dsplits > 1 ? typed<float>(&dpo) : nullptr, *dpmf = dsplits > 1 ? typed<float>(&dpm) : nullptr;
  const int32_t *tb = typed<int32_t>(tables), *sq = typed<int32_t>(seq), *ps = typed<int32_t>(pos), *tl = typed<int32_t>(tiles);
  const int64_t k0 = k->stride(0), k1 = k->stride(1), k2 = k->stride(2), v0 = v->stride(0), v2 = v->stride(2), v3 = v->stride(3);
  const float *sk = typed<float>(sinks), *sl = typed<float>(slopes), *gt = typed<float>(gate);
  // both in one launch (attn_step_kernel), unless the decoding part's chunks are for fewer waves than the prompts' tiles (24 heads of 128, 64 requests of 2,048
  // keys for four waves beside 1,500 tokens for eight: 111 us in two launches, 125 in one)
  if (lead && splits == 1 && first == lead && page % 32 == 0 && dwaves >= waves && (hd == 64 || (hd == 128 && !general)) && tile_tokens <= 2 * per_wave &&
      !TS_REFUSED("paged_attention_step",
                  ts_paged_attention_step(ptr(&out), dpof, dpmf, ptr(q), ptr(k), ptr(v), tb, sq, ps, lead, dsplits, dchunk, dwaves, tl, tiles->size(0), tile_tokens, waves,
                                          nh, nkv, hd, page, k0, k1, k2, v0, v2, v3, blocks, scale, window, run, general, softcap, sink, sk, sl, gt, gstride, stream())))
    return wrap(out);
  if (lead && general) {
    if (TS_REFUSED("paged_attention_decode_general",
                   ts_paged_attention_decode_general(ptr(&out), dpof, dpmf, ptr(q), ptr(k), ptr(v), tb, sq, ps, lead, nh, nkv, hd, page, k0, k1, k2, v0, v2, v3, blocks,
                                                     dsplits, dchunk, dwaves, scale, window, run, softcap, sink, sk, sl, gt, gstride, stream())))
      return none();
  } else if (lead) {
    if (TS_REFUSED("paged_attention_decode", ts_paged_attention_decode(ptr(&out), dpof, dpmf, ptr(q), ptr(k), ptr(v), tb, sq, ps, lead, nh, nkv, hd, page, k0, k1, k2, v0,
                                                                       v2, v3, blocks, dsplits, dchunk, dwaves, scale, window, run, 1, stream())))
      return none();
  }
  const bool behind = lead > 0;
  if (general) {
    if (TS_REFUSED("paged_attention_prefill_general",
                   ts_paged_attention_prefill_general(ptr(&out), ptr(q), ptr(k), ptr(v), tb, sq, ps, tl, tiles->size(0), tile_tokens, waves, nh, nkv, hd, page, k0, k1,
                                                      k2, v0, v2, v3, blocks, scale, window, first, T, splits, chunk, pof, pmf, run, softcap, sink, sk, sl, gt, gstride,
                                                      stream()), behind))
      return none();
  } else if (TS_REFUSED("paged_attention_prefill",
                        ts_paged_attention_prefill(ptr(&out), ptr(q), ptr(k), ptr(v), tb, sq, ps, tl, tiles->size(0), tile_tokens, waves, nh, nkv, hd, page, k0, k1, k2, v0,
                                                   v2, v3, blocks, scale, window, first, T, splits, chunk, pof, pmf, run, stream()), behind)) {
    return none();
  }
  return wrap(out);
}

// ---- units ----

PyObject* capped_glu(Args a) {      // gate|up, limit, slope, up_shift, out code, form's number -> y
  const Tensor* x = a.tensor();
  const float limit = a.number(), slope = a.number(), shift = a.number();
  const int out_code = a.i32(), act = a.i32();
  if (!a.done() || out_code < 0 || out_code > 1 || code(*x) < 0 || x->dim() != 2 || x->size(1) % 2 || x->stride(1) != 1 || x->stride(0) < x->size(1)) return none();
  if (!fits(x->size(0)) || !fits(x->size(1))) return none();
  Tensor y = make(*x, {x->size(0), x->size(1) / 2}, out_code ? at::kBFloat16 : at::kFloat);
  if (TS_REFUSED("capped_glu",
                 ts_capped_glu(ptr(&y), out_code, ptr(x), code(*x), x->stride(0), x->size(0), x->size(1) / 2, limit, slope, shift, act, stream())))
    return none();
  return wrap(y);
}

PyObject* mlstm_finish(Args a) {      // o, weight, gate, heads, value size, eps, out code, silu -> rows
  const Tensor *o = a.tensor(), *w = a.maybe(), *g = a.tensor();
  const int heads = a.i32(), vdim = a.i32();
  const float eps = a.number();
  const int out_code = a.i32(), silu = a.i32();
  if (!a.done() || out_code < 0 || out_code > 1 || !f32(*o) || o->dim() != 2 || !o->is_contiguous() || heads <= 0 || vdim <= 0) return none();
  const int64_t T = o->size(0), width = (int64_t)heads * vdim;
  if (o->size(1) != width || !fits(T) || !fits(width) || (w && !vector(*w, at::kFloat, width) && !vector(*w, at::kFloat, vdim))) return none();
  if (!f32(*g) || !matrix(*g, T, width) || g->stride(1) != 1 || g->stride(0) < width) return none();
  Tensor y = make(*o, {T, width}, out_code ? at::kBFloat16 : at::kFloat);
  if (TS_REFUSED("mlstm_finish",
                 ts_mlstm_finish(ptr(&y), out_code, typed<float>(o), typed<float>(w), typed<float>(g), g->stride(0), T, heads, vdim, eps, w && w->size(0) ==
                                 width ? vdim : 0, silu, stream())))
    return none();
  return wrap(y);
}

template <PyObject* (*F)(Args)> PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  return F(Args{args, n});
  END_HANDLE_TH_ERRORS
}

#define TS_CALL(NAME) {#NAME, (PyCFunction)(void (*)())entry<NAME>, METH_FASTCALL, nullptr}
PyMethodDef calls[] = {TS_CALL(rmsnorm),
                       TS_CALL(stream_post_norm),
                       TS_CALL(stream_update_norm),
                       TS_CALL(gemm_library),
                       TS_CALL(gemm_slices),
                       TS_CALL(gemm_glu),
                       TS_CALL(gemm_rows64),
                       TS_CALL(gemm_rows64_sliced),
                       TS_CALL(rope_store),
                       TS_CALL(qkv_rope_store_sliced),
                       TS_CALL(qkv_finish),
                       TS_CALL(attention_step),
                       TS_CALL(capped_glu),
                       TS_CALL(mlstm_finish),
                       {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "tinyserve_hip_calls", nullptr, -1, calls, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_tinyserve_hip_calls() { return PyModule_Create(&module); }
