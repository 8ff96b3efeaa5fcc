// The regular calls of engine.kernels, from Python arguments to the kernels'
// C entry points in one native step.
//
// The Python wrappers accept many forms of argument (other dtypes, strided
// tensors, indices on the host, ...), which costs 15-25 us of interpreter
// time per call: more than a decode step's kernels take.  Each function here
// takes the same tensors, handles exactly the form that needs no conversion or
// copy, allocates the outputs and launches; for anything else it returns None
// without having done anything, and the wrapper goes its general way, which
// converts, copies or raises.  Nothing is kept between calls.
// (Measured, eager calls back to back: one decode step of the whole layer at
// B = 1 / 64 108 / 113 us through the wrappers, 31 / 78 us here, of which 24 / 76
// are kernels; a decode recurrence at B = 1 16.1 and 5.7 us.)
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>
#include <limits>

#include "gdn_capi.h"
#include "gdn_gate_proj.h"

namespace {

// The library's entry points, from the copy that the ctypes binding loaded.
struct Entries {
  decltype(&gdn_last_error_string) last_error;
  decltype(&gdn_recurrent_fwd) recurrent;
  decltype(&gdn_recurrent_fwd_gated) recurrent_gated;
  decltype(&gdn_chunk_fwd) chunk;
  decltype(&gdn_chunk_fwd_gated) chunk_gated;
  decltype(&gdn_chunk_workspace_bytes) chunk_workspace;
  decltype(&gdn_rmsnorm_gated_fwd) rmsnorm;
  decltype(&gdn_in_proj_decode) in_proj;
  decltype(&gdn_out_proj_workspace_bytes) out_proj_workspace;
  decltype(&gdn_out_proj_decode) out_proj;
  decltype(&causal_conv1d_fwd) conv;
  decltype(&gdn_gate_proj) gate_proj;
} fn;

using at::Tensor;

// An argument's tensor: a plain torch.Tensor or Parameter on a GPU.  `ok` turns
// false for any other object (None is an absent tensor).
const Tensor *tensor(PyObject *o, bool &ok) {
  if (o == Py_None) return nullptr;
  if (!THPVariable_CheckExact(o)) {
    ok = false;
    return nullptr;
  }
  const Tensor &t = THPVariable_Unpack(o);
  if (!t.is_cuda() || t.layout() != at::kStrided) ok = false;
  return &t;
}
bool same_device(const Tensor &ref, std::initializer_list<const Tensor *> ts) {
  for (const Tensor *t : ts)
    if (t && t->device() != ref.device()) return false;
  return true;
}
int dtype_code(const Tensor &t) {
  switch (t.scalar_type()) {
    case at::kFloat: return GDN_DTYPE_F32;
    case at::kBFloat16: return GDN_DTYPE_BF16;
    case at::kHalf: return GDN_DTYPE_F16;
    default: return -1;
  }
}
bool fits32(int64_t x) { return x >= 0 && x <= std::numeric_limits<int32_t>::max(); }
void *ptr(const Tensor *t) { return t ? t->data_ptr() : nullptr; }
int64_t rows(const Tensor *t) { return t ? t->size(0) : 0; }
bool index_ok(const Tensor *t) { return !t || (t->scalar_type() == at::kLong && t->is_contiguous()); }
void *stream_of(const Tensor &t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
Tensor empty(at::IntArrayRef sizes, const Tensor &like) { return at::empty(sizes, like.options().requires_grad(false)); }
Tensor empty(at::IntArrayRef sizes, const Tensor &like, at::ScalarType dt) {
  return at::empty(sizes, like.options().dtype(dt).requires_grad(false));
}

// [B, T, H, D] as a token-major stream: its token stride, or -1.
int64_t token_stride(const Tensor &x) {
  const int64_t b = x.size(0), t = x.size(1), h = x.size(2), d = x.size(3);
  const int64_t st = t > 1 ? x.stride(1) : b > 1 ? x.stride(0) : h * d;
  const bool ok = x.stride(3) == 1 && (h == 1 || x.stride(2) == d) && st >= h * d && st % 8 == 0 &&
                  (b == 1 || x.stride(0) == t * st) && x.storage_offset() % 8 == 0;
  return ok ? st : -1;
}
// [B, T, H] per-token rows: their token stride, or -1.
int64_t gate_stride(const Tensor &x, int64_t b, int64_t t, int64_t h) {
  if (x.dim() != 3 || x.size(0) != b || x.size(1) != t || x.size(2) != h) return -1;
  const int64_t st = t > 1 ? x.stride(1) : b > 1 ? x.stride(0) : h;
  const bool ok = (x.stride(2) == 1 || h == 1) && st >= h && (b == 1 || x.stride(0) == t * st);
  return ok ? st : -1;
}

PyObject *failed(const char *what, int status) {
  return PyErr_Format(PyExc_RuntimeError, "%s failed (status %d): %s", what, status, fn.last_error());
}
PyObject *none() { Py_RETURN_NONE; }

// Other Python threads run while this one allocates and launches (the
// arguments stay alive in the caller's frame).
struct NoGil {
  PyThreadState *state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
};

// q, k, v and the gates of a recurrence or chunk call.
struct Core {
  const Tensor *q, *k, *v, *ga, *gb, *alog, *dtb, *state, *idx, *cu;
  int64_t b, t, hk, hv, dk, dv, qs, ks, vs, gs, n_seqs;
  int dt, gdt;
  float scale;
  int l2norm;

  // args: q k v gate0 gate1 A_log dt_bias scale l2norm state idx cu
  bool read(PyObject *const *a) {
    bool ok = true;
    q = tensor(a[0], ok), k = tensor(a[1], ok), v = tensor(a[2], ok), ga = tensor(a[3], ok), gb = tensor(a[4], ok);
    alog = tensor(a[5], ok), dtb = tensor(a[6], ok), state = tensor(a[9], ok), idx = tensor(a[10], ok);
    cu = tensor(a[11], ok);
    if (!ok || !q || !k || !v || !ga || !gb || !alog != !dtb) return false;
    if (!same_device(*q, {k, v, ga, gb, alog, dtb, state, idx, cu})) return false;
    if (q->dim() != 4 || v->dim() != 4 || k->sizes() != q->sizes()) return false;
    b = q->size(0), t = q->size(1), hk = q->size(2), dk = q->size(3), hv = v->size(2), dv = v->size(3);
    if (v->size(0) != b || v->size(1) != t || b < 1 || t < 1 || hk < 1 || hv < 1 || hv % hk || dk < 1 || dv < 1) return false;
    dt = dtype_code(*q);
    if (dt < 0 || k->scalar_type() != q->scalar_type() || v->scalar_type() != q->scalar_type()) return false;
    qs = token_stride(*q), ks = token_stride(*k), vs = token_stride(*v);
    if (qs < 0 || ks < 0 || vs < 0) return false;
    gs = gate_stride(*ga, b, t, hv);
    if (gs < 0 || gate_stride(*gb, b, t, hv) != gs) return false;
    gdt = dtype_code(*gb);
    if (gdt < 0) return false;
    if (alog) {  // raw projections
      if (ga->scalar_type() != gb->scalar_type()) return false;
      for (const Tensor *x : {alog, dtb})
        if (x->scalar_type() != at::kFloat || !x->is_contiguous() || x->numel() != hv) return false;
    } else if (ga->scalar_type() != at::kFloat || gs != hv) {
      return false;
    }
    if (cu && (cu->scalar_type() != at::kInt || !cu->is_contiguous() || cu->numel() < 2 || b != 1)) return false;
    n_seqs = cu ? cu->numel() - 1 : b;
    if (!fits32(n_seqs) || !fits32(b * t)) return false;
    if (!index_ok(idx) || (idx && (!state || idx->numel() < n_seqs))) return false;
    if (state && (state->dim() != 4 || state->scalar_type() != at::kFloat || !state->is_contiguous() ||
                  state->size(1) != hv || state->size(2) != dk || state->size(3) != dv ||
                  (!idx && state->size(0) != n_seqs)))
      return false;
    if (a[7] == Py_None) {
      scale = static_cast<float>(1.0 / std::sqrt(static_cast<double>(dk)));
    } else {
      if (!PyFloat_CheckExact(a[7])) return false;
      scale = static_cast<float>(PyFloat_AS_DOUBLE(a[7]));
    }
    if (!PyBool_Check(a[8])) return false;
    l2norm = a[8] == Py_True;
    return true;
  }
  int T() const { return static_cast<int>(cu ? b * t : t); }

  int run_recurrent(const Tensor *in, const Tensor *in_idx, const Tensor *out, const Tensor *out_idx, const Tensor &o,
                    const Tensor *snap) const {
    const auto i64 = [](const Tensor *x) { return static_cast<const int64_t *>(ptr(x)); };
    const auto f32 = [](const Tensor *x) { return static_cast<float *>(ptr(x)); };
    const auto cu32 = static_cast<const int32_t *>(ptr(cu));
    if (alog)
      return fn.recurrent_gated(ptr(q), ptr(k), ptr(v), dt, qs, ks, vs, ptr(ga), ptr(gb), gdt, gs, f32(alog), f32(dtb),
                                f32(in), i64(in_idx), rows(in), f32(out), i64(out_idx), rows(out), o.data_ptr(), dt,
                                f32(snap), cu32, n_seqs, T(), hk, hv, dk, dv, scale, l2norm, stream_of(*q));
    return fn.recurrent(ptr(q), ptr(k), ptr(v), dt, qs, ks, vs, f32(ga), ptr(gb), gdt, f32(in), i64(in_idx), rows(in),
                        f32(out), i64(out_idx), rows(out), o.data_ptr(), dt, f32(snap), cu32, n_seqs, T(), hk, hv, dk,
                        dv, scale, l2norm, stream_of(*q));
  }
  int run_chunk(const Tensor *in, const Tensor *in_idx, const Tensor *out, const Tensor *out_idx, const Tensor &o,
                const Tensor &ws, size_t ws_bytes) const {
    const auto i64 = [](const Tensor *x) { return static_cast<const int64_t *>(ptr(x)); };
    const auto f32 = [](const Tensor *x) { return static_cast<float *>(ptr(x)); };
    const auto cu32 = static_cast<const int32_t *>(ptr(cu));
    if (alog)
      return fn.chunk_gated(ptr(q), ptr(k), ptr(v), dt, qs, ks, vs, ptr(ga), ptr(gb), gdt, gs, f32(alog), f32(dtb),
                            f32(in), i64(in_idx), rows(in), f32(out), i64(out_idx), rows(out), o.data_ptr(), dt, cu32,
                            n_seqs, T(), hk, hv, dk, dv, scale, l2norm, ws.data_ptr(), ws_bytes, stream_of(*q));
    return fn.chunk(ptr(q), ptr(k), ptr(v), dt, qs, ks, vs, f32(ga), ptr(gb), gdt, f32(in), i64(in_idx), rows(in),
                    f32(out), i64(out_idx), rows(out), o.data_ptr(), dt, cu32, n_seqs, T(), hk, hv, dk, dv, scale,
                    l2norm, ws.data_ptr(), ws_bytes, stream_of(*q));
  }
};

// (o, final state): `state` itself when updated in place.
PyObject *pair(const Tensor &o, PyObject *state, bool inplace, const Tensor &made) {
  PyObject *r = PyTuple_New(2);
  if (!r) return nullptr;
  PyTuple_SET_ITEM(r, 0, THPVariable_Wrap(o));
  PyObject *s = inplace ? Py_NewRef(state) : made.defined() ? THPVariable_Wrap(made) : Py_NewRef(Py_None);
  PyTuple_SET_ITEM(r, 1, s);
  return r;
}

// recurrent(q, k, v, gate0, gate1, A_log, dt_bias, scale, l2norm, state, idx, cu, inplace, output_final, snapshots)
PyObject *recurrent(PyObject *, PyObject *const *a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Core c;
  bool ok = true;
  if (n != 15 || !c.read(a) || !PyBool_Check(a[12]) || !PyBool_Check(a[13])) return none();
  const bool inplace = a[12] == Py_True, output = a[13] == Py_True;
  const Tensor *snap = tensor(a[14], ok);
  if (!ok || (inplace && !c.state)) return none();
  if (snap && (snap->scalar_type() != at::kFloat || !snap->is_contiguous() || !same_device(*c.q, {snap}) ||
               snap->sizes() != at::IntArrayRef({c.n_seqs, c.t, c.hv, c.dk, c.dv})))
    return none();
  Tensor o, made;
  int st;
  {
    NoGil unlocked;
    o = empty({c.b, c.t, c.hv, c.dv}, *c.q);
    if (output && !inplace) made = empty({c.n_seqs, c.hv, c.dk, c.dv}, *c.q, at::kFloat);
    const Tensor *out = inplace ? c.state : made.defined() ? &made : nullptr;
    st = c.run_recurrent(c.state, c.idx, out, inplace ? c.idx : nullptr, o, snap);
  }
  if (st) return failed(c.alog ? "gdn_recurrent_fwd_gated" : "gdn_recurrent_fwd", st);
  return pair(o, a[9], inplace, made);
  END_HANDLE_TH_ERRORS
}

// chunk(q, k, v, gate0, gate1, A_log, dt_bias, scale, l2norm, state, idx, cu, inplace, output_final, read_idx):
// read_idx None: the initial states come through idx.
PyObject *chunk(PyObject *, PyObject *const *a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Core c;
  bool ok = true;
  if (n != 15 || !c.read(a) || !PyBool_Check(a[12]) || !PyBool_Check(a[13])) return none();
  const bool inplace = a[12] == Py_True, output = a[13] == Py_True;
  const Tensor *rd = tensor(a[14], ok);
  if (!ok || (inplace && !c.state)) return none();
  if (rd && (!c.state || !index_ok(rd) || rd->numel() < c.n_seqs || !same_device(*c.q, {rd}))) return none();
  const bool chunked = c.dt == GDN_DTYPE_BF16 && c.dk == 128 && c.dv == 128;
  Tensor o, made;
  int st;
  {
    NoGil unlocked;
    o = empty({c.b, c.t, c.hv, c.dv}, *c.q);
    if (output && !inplace) made = empty({c.n_seqs, c.hv, c.dk, c.dv}, *c.q, at::kFloat);
    const Tensor *out = inplace ? c.state : made.defined() ? &made : nullptr;
    const Tensor *in_idx = rd ? rd : c.idx, *out_idx = inplace ? c.idx : nullptr;
    if (chunked) {
      const size_t bytes = fn.chunk_workspace(c.n_seqs, c.b * c.t, c.hv, c.dk, c.dv);
      const Tensor ws = empty({static_cast<int64_t>(bytes ? bytes : 1)}, *c.q, at::kByte);
      st = c.run_chunk(c.state, in_idx, out, out_idx, o, ws, bytes);
    } else {
      st = c.run_recurrent(c.state, in_idx, out, out_idx, o, nullptr);
    }
  }
  if (st && chunked) return failed(c.alog ? "gdn_chunk_fwd_gated" : "gdn_chunk_fwd", st);
  if (st) return failed(c.alog ? "gdn_recurrent_fwd_gated" : "gdn_recurrent_fwd", st);
  return pair(o, a[9], inplace, made);
  END_HANDLE_TH_ERRORS
}

bool norm_weight_ok(const Tensor &w, int64_t d) {
  return dtype_code(w) >= 0 && w.is_contiguous() && w.numel() == d && reinterpret_cast<uintptr_t>(w.data_ptr()) % 32 == 0;
}

// rms_norm(x, z, weight, eps): x and z contiguous, the result in x's dtype
PyObject *rms_norm(PyObject *, PyObject *const *a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  bool ok = true;
  if (n != 4 || !PyFloat_CheckExact(a[3])) return none();
  const Tensor *x = tensor(a[0], ok), *z = tensor(a[1], ok), *w = tensor(a[2], ok);
  if (!ok || !x || !z || !w || !same_device(*x, {z, w}) || x->dim() < 2 || x->sizes() != z->sizes()) return none();
  const int64_t d = x->size(-1), h = x->size(-2);
  if (x->numel() == 0 || !x->is_contiguous() || !z->is_contiguous() || dtype_code(*x) < 0 || dtype_code(*z) < 0 ||
      x->storage_offset() % 8 || z->storage_offset() % 8 || (h * d) % 8 || !norm_weight_ok(*w, d) || !fits32(h))
    return none();
  const float eps = static_cast<float>(PyFloat_AS_DOUBLE(a[3]));
  Tensor y;
  int st;
  {
    NoGil unlocked;
    y = empty(x->sizes(), *x);
    st = fn.rmsnorm(x->data_ptr(), dtype_code(*x), h * d, z->data_ptr(), dtype_code(*z), h * d, w->data_ptr(),
                    dtype_code(*w), y.data_ptr(), dtype_code(y), h * d, x->numel() / (h * d), h, d, eps, stream_of(*x));
  }
  if (st) return failed("gdn_rmsnorm_gated_fwd", st);
  return THPVariable_Wrap(y);
  END_HANDLE_TH_ERRORS
}

bool bf16_matrix(const Tensor *w, int64_t k) {  // an nn.Linear weight that the kernels read in place
  return w && w->scalar_type() == at::kBFloat16 && w->dim() == 2 && w->size(1) == k && w->is_contiguous() &&
         reinterpret_cast<uintptr_t>(w->data_ptr()) % 16 == 0;
}
// bf16 rows [M, K] or [M, 1, K]: their row stride, or -1
int64_t decode_rows(const Tensor &x, int64_t &m, int64_t &k) {
  if (x.scalar_type() != at::kBFloat16 || (x.dim() != 2 && x.dim() != 3) || (x.dim() == 3 && x.size(1) != 1)) return -1;
  m = x.size(0), k = x.size(-1);
  if (m < 1 || x.stride(-1) != 1 || x.stride(0) % 8 || reinterpret_cast<uintptr_t>(x.data_ptr()) % 16) return -1;
  return m > 1 ? x.stride(0) : k;
}

// The operands of gdn_in_proj_decode.
struct InProj {
  const Tensor *x, *w[4], *cw, *cb, *pool, *idx;
  int64_t m, k, xs, n[4];
  // args: hidden w_qkv w_z w_b w_a conv_weight conv_bias pool idx
  bool read(PyObject *const *a) {
    bool ok = true;
    x = tensor(a[0], ok);
    for (int i = 0; i < 4; ++i) w[i] = tensor(a[1 + i], ok);
    cw = tensor(a[5], ok), cb = tensor(a[6], ok), pool = tensor(a[7], ok), idx = tensor(a[8], ok);
    if (!ok || !x || !cw || !pool || !same_device(*x, {w[0], w[1], w[2], w[3], cw, cb, pool, idx})) return false;
    xs = decode_rows(*x, m, k);
    if (xs < 0 || (k != 1024 && k != 2048)) return false;
    for (int i = 0; i < 4; ++i) {
      if (!bf16_matrix(w[i], k)) return false;
      n[i] = w[i]->size(0);
    }
    if (n[0] % 64 || n[1] % 64 || n[2] % 4 || n[3] % 4 || n[2] > 32 || n[3] > 32 || !n[0] || !n[1] || !n[2] || !n[3])
      return false;
    if (cw->scalar_type() != at::kBFloat16 || !cw->is_contiguous() || cw->size(0) != n[0] || cw->numel() != n[0] * 4) return false;
    if (cb && (cb->scalar_type() != at::kBFloat16 || !cb->is_contiguous() || cb->numel() != n[0])) return false;
    if (pool->scalar_type() != at::kBFloat16 || pool->dim() != 3 || pool->size(1) != n[0] || pool->size(2) != 4 ||
        !pool->is_contiguous())
      return false;
    return index_ok(idx) && (idx ? idx->numel() == m : true) && fits32(m);
  }
  int run(Tensor (&out)[4], int silu) const {
    for (int i = 0; i < 4; ++i) out[i] = empty({m, n[i]}, *x);
    return fn.in_proj(x->data_ptr(), xs, ptr(w[0]), ptr(w[1]), ptr(w[2]), ptr(w[3]), m, k, n[0], n[1], n[2], n[3],
                      cw->data_ptr(), ptr(cb), pool->data_ptr(), static_cast<const int64_t *>(ptr(idx)), pool->size(0),
                      out[0].data_ptr(), out[1].data_ptr(), out[2].data_ptr(), out[3].data_ptr(), silu, stream_of(*x));
  }
};

// in_proj(hidden, w_qkv, w_z, w_b, w_a, conv_weight, conv_bias, pool, idx, silu)
PyObject *in_proj(PyObject *, PyObject *const *a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  InProj p;
  if (n != 10 || !PyBool_Check(a[9]) || !p.read(a)) return none();
  const int silu = a[9] == Py_True;
  Tensor out[4];
  int st;
  {
    NoGil unlocked;
    st = p.run(out, silu);
  }
  if (st) return failed("gdn_in_proj_decode", st);
  PyObject *r = PyTuple_New(4);
  if (!r) return nullptr;
  for (int i = 0; i < 4; ++i) PyTuple_SET_ITEM(r, i, THPVariable_Wrap(out[i]));
  return r;
  END_HANDLE_TH_ERRORS
}

bool out_proj_ok(int64_t k, int64_t n) { return k % 512 == 0 && k > 0 && k <= 8192 && n % 64 == 0 && n > 0; }
int run_out_proj(const void *x, int64_t xs, const Tensor &w, int64_t m, int64_t k, const Tensor &y, const Tensor &like) {
  const int64_t n = w.size(0);
  const int64_t bytes = static_cast<int64_t>(fn.out_proj_workspace(m, k, n));
  const Tensor ws = empty({bytes > 16 ? bytes : 16}, like, at::kByte);
  return fn.out_proj(x, xs, w.data_ptr(), m, k, n, y.data_ptr(), n, ws.data_ptr(), ws.numel(), stream_of(like));
}

// out_proj(x, weight)
PyObject *out_proj(PyObject *, PyObject *const *a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  bool ok = true;
  if (n != 2) return none();
  const Tensor *x = tensor(a[0], ok), *w = tensor(a[1], ok);
  int64_t m, k;
  if (!ok || !x || !w || !same_device(*x, {w})) return none();
  const int64_t xs = decode_rows(*x, m, k);
  if (xs < 0 || !bf16_matrix(w, k) || !out_proj_ok(k, w->size(0)) || !fits32(m)) return none();
  Tensor y;
  int st;
  {
    NoGil unlocked;
    y = x->dim() == 3 ? empty({m, 1, w->size(0)}, *x) : empty({m, w->size(0)}, *x);
    st = run_out_proj(x->data_ptr(), xs, *w, m, k, y, *x);
  }
  if (st) return failed("gdn_out_proj_decode", st);
  return THPVariable_Wrap(y);
  END_HANDLE_TH_ERRORS
}

// gate_proj(hidden, w_b, w_a): hidden [..., K] contiguous bf16; (b, a), each [..., n]
PyObject *gate_proj(PyObject *, PyObject *const *a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  bool ok = true;
  if (n != 3) return none();
  const Tensor *x = tensor(a[0], ok), *wb = tensor(a[1], ok), *wa = tensor(a[2], ok);
  if (!ok || !x || !wb || !wa || !same_device(*x, {wb, wa})) return none();
  if (x->scalar_type() != at::kBFloat16 || x->dim() < 2 || x->numel() == 0 || !x->is_contiguous() ||
      reinterpret_cast<uintptr_t>(x->data_ptr()) % 16)
    return none();
  const int64_t k = x->size(-1), m = x->numel() / k;
  if (!bf16_matrix(wb, k) || !bf16_matrix(wa, k) || !fits32(m)) return none();
  const int64_t cols = wb->size(0);
  if (wa->size(0) != cols || (cols != 16 && cols != 32) || (k != 1024 && k != 2048)) return none();
  Tensor out[2];
  int st;
  {
    NoGil unlocked;
    auto sizes = x->sizes().vec();
    sizes.back() = cols;
    for (Tensor &t : out) t = empty(sizes, *x);
    st = fn.gate_proj(x->data_ptr(), wb->data_ptr(), wa->data_ptr(), m, k, cols, out[0].data_ptr(), out[1].data_ptr(),
                      stream_of(*x));
  }
  if (st) return failed("gdn_gate_proj", st);
  PyObject *r = PyTuple_New(2);
  if (!r) return nullptr;
  for (int i = 0; i < 2; ++i) PyTuple_SET_ITEM(r, i, THPVariable_Wrap(out[i]));
  return r;
  END_HANDLE_TH_ERRORS
}

// conv(x, weight, bias, silu, pool, idx, read_idx, cu): x [tokens, C], or [B, C, T] with the channels
// contiguous, in the weight's dtype; read_idx None: the history comes through idx.  Returns y laid out as x.
PyObject *conv(PyObject *, PyObject *const *a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  bool ok = true;
  if (n != 8 || !PyBool_Check(a[3])) return none();
  const Tensor *x = tensor(a[0], ok), *w = tensor(a[1], ok), *bias = tensor(a[2], ok), *pool = tensor(a[4], ok);
  const Tensor *idx = tensor(a[5], ok), *rd = tensor(a[6], ok), *cu = tensor(a[7], ok);
  if (!ok || !x || !w || !same_device(*x, {w, bias, pool, idx, rd, cu})) return none();
  const auto dt = x->scalar_type();
  if (dtype_code(*x) < 0 || x->numel() == 0 || (x->dim() != 2 && x->dim() != 3)) return none();
  const bool bct = x->dim() == 3;
  const int64_t b = bct ? x->size(0) : 1, c = x->size(1), t = bct ? x->size(2) : x->size(0);
  const int64_t sb = bct ? x->stride(0) : 0, sc = x->stride(1), stt = bct ? x->stride(2) : x->stride(0);
  const int64_t st = t > 1 ? stt : b > 1 ? sb : c;
  if (sc != 1 || st % 8 || x->storage_offset() % 8 || (b > 1 && t > 1 && sb != t * st)) return none();
  if (w->scalar_type() != dt || !w->is_contiguous() || w->dim() != 2 || w->size(0) != c) return none();
  if (bias && (bias->scalar_type() != dt || !bias->is_contiguous() || bias->numel() != c)) return none();
  if (cu && (cu->scalar_type() != at::kInt || !cu->is_contiguous() || cu->numel() < 2 || b != 1)) return none();
  const int64_t n_seqs = cu ? cu->numel() - 1 : b;
  if (!fits32(n_seqs) || !fits32(b * t) || !index_ok(idx) || !index_ok(rd)) return none();
  int64_t s_len = w->size(1) > 1 ? 4 : 3;
  if (pool) {
    if (pool->scalar_type() != dt || pool->dim() != 3 || !pool->is_contiguous() || pool->size(1) != c) return none();
    if (idx ? idx->numel() < n_seqs : pool->size(0) != n_seqs) return none();
    s_len = pool->size(2);
  } else if (idx) {
    return none();
  }
  if (rd && (!pool || rd->numel() < n_seqs)) return none();
  const int silu = a[3] == Py_True;
  const auto i64 = [](const Tensor *q) { return static_cast<const int64_t *>(ptr(q)); };
  Tensor y;
  int status;
  {
    NoGil unlocked;
    y = empty({b, t, c}, *x);
    status = fn.conv(x->data_ptr(), st, w->data_ptr(), ptr(bias), y.data_ptr(), c, ptr(pool), i64(rd ? rd : idx),
                     rows(pool), ptr(pool), i64(idx), rows(pool), static_cast<const int32_t *>(ptr(cu)), n_seqs,
                     cu ? b * t : t, c, w->size(1), s_len, silu, dtype_code(*x), stream_of(*x));
  }
  if (status) return failed("causal_conv1d_fwd", status);
  return THPVariable_Wrap(bct ? y.transpose(1, 2) : y.view({t, c}));
  END_HANDLE_TH_ERRORS
}

// core_decode(qkv [B, C], z [B, value_dim], b, a [B, Hv], slots, key_dim, value_dim, head_k_dim, head_v_dim, A_log,
// dt_bias, state_pool, norm_weight, eps): between a decode step's projections, the recurrence on slot
// pools and the gated norm; [B, 1, value_dim]
PyObject *core_decode(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  bool ok = true;
  if (n != 14 || !PyFloat_CheckExact(args[13])) return none();
  int64_t dims[4];
  for (int i = 0; i < 4; ++i) {
    if (!PyLong_CheckExact(args[5 + i])) return none();
    dims[i] = PyLong_AsLongLong(args[5 + i]);
  }
  if (PyErr_Occurred()) return nullptr;
  const int64_t key = dims[0], val = dims[1], dk = dims[2], dv = dims[3];
  const Tensor *qkv = tensor(args[0], ok), *z = tensor(args[1], ok), *b = tensor(args[2], ok), *a = tensor(args[3], ok);
  const Tensor *slots = tensor(args[4], ok), *alog = tensor(args[9], ok), *dtb = tensor(args[10], ok);
  const Tensor *state = tensor(args[11], ok), *nw = tensor(args[12], ok);
  if (!ok || !qkv || !z || !b || !a || !slots || !alog || !dtb || !state || !nw) return none();
  if (!same_device(*qkv, {z, b, a, slots, alog, dtb, state, nw})) return none();
  if (key < 1 || val < 1 || dk < 1 || dv < 1 || key % dk || val % dv) return none();
  const int64_t hk = key / dk, hv = val / dv, m = qkv->size(0), c = 2 * key + val;
  if (hv % hk || dk % 8 || dv % 8 || !fits32(m) || m < 1) return none();
  const auto rows_of = [&](const Tensor *x, int64_t w) {
    return x->scalar_type() == at::kBFloat16 && x->dim() == 2 && x->size(0) == m && x->size(1) == w && x->is_contiguous() &&
           x->storage_offset() % 8 == 0;
  };
  if (!rows_of(qkv, c) || !rows_of(z, val) || !rows_of(b, hv) || !rows_of(a, hv)) return none();
  if (!index_ok(slots) || slots->numel() != m) return none();
  for (const Tensor *x : {alog, dtb})
    if (x->scalar_type() != at::kFloat || !x->is_contiguous() || x->numel() != hv) return none();
  if (state->dim() != 4 || state->scalar_type() != at::kFloat || !state->is_contiguous() || state->size(1) != hv ||
      state->size(2) != dk || state->size(3) != dv || !norm_weight_ok(*nw, dv))
    return none();
  const float eps = static_cast<float>(PyFloat_AS_DOUBLE(args[13]));
  const char *what = "gdn_recurrent_fwd_gated";
  Tensor normed;
  int st;
  {
    NoGil unlocked;
    void *stream = stream_of(*qkv);
    const Tensor core = empty({m, val}, *qkv);
    normed = empty({m, 1, val}, *qkv);
    auto *y = static_cast<char *>(qkv->data_ptr());
    const auto *ids = static_cast<const int64_t *>(slots->data_ptr());
    auto *pool = static_cast<float *>(state->data_ptr());
    st = fn.recurrent_gated(y, y + 2 * key, y + 4 * key, GDN_DTYPE_BF16, c, c, c, a->data_ptr(), b->data_ptr(),
                            GDN_DTYPE_BF16, hv, static_cast<const float *>(alog->data_ptr()),
                            static_cast<const float *>(dtb->data_ptr()), pool, ids, state->size(0), pool, ids,
                            state->size(0), core.data_ptr(), GDN_DTYPE_BF16, nullptr, nullptr, m, 1, hk, hv, dk, dv,
                            static_cast<float>(1.0 / std::sqrt(static_cast<double>(dk))), 1, stream);
    if (!st) {
      what = "gdn_rmsnorm_gated_fwd";
      st = fn.rmsnorm(core.data_ptr(), GDN_DTYPE_BF16, val, z->data_ptr(), GDN_DTYPE_BF16, val, nw->data_ptr(),
                      dtype_code(*nw), normed.data_ptr(), GDN_DTYPE_BF16, val, m, hv, dv, eps, stream);
    }
  }
  if (st) return failed(what, st);
  return THPVariable_Wrap(normed);
  END_HANDLE_TH_ERRORS
}

// bind(addresses): the library's entry points, in Entries' order
PyObject *bind(PyObject *, PyObject *const *a, Py_ssize_t n) {
  constexpr int N = sizeof(Entries) / sizeof(void *);
  if (n != N) return PyErr_Format(PyExc_TypeError, "bind takes %d addresses", N);
  void *addr[N];
  for (int i = 0; i < N; ++i) {
    addr[i] = PyLong_AsVoidPtr(a[i]);
    if (PyErr_Occurred()) return nullptr;
  }
  static_assert(sizeof(addr) == sizeof(fn), "Entries holds function pointers only");
  __builtin_memcpy(&fn, addr, sizeof(fn));
  Py_RETURN_NONE;
}

#define GDN_METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {GDN_METHOD(bind),    GDN_METHOD(recurrent), GDN_METHOD(chunk),
                         GDN_METHOD(rms_norm), GDN_METHOD(in_proj),   GDN_METHOD(out_proj),
                         GDN_METHOD(conv),     GDN_METHOD(core_decode), GDN_METHOD(gate_proj), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_gdn_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__gdn_host(void) { return PyModule_Create(&module); }
