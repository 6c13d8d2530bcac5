// Native bindings of the operations an eager prefill launches one by one: the argument checks
// of needle_amd/ops.py and the launch, without the interpreter between them.
//
// ops.py is the definition: every function here returns None for a call it does not take as it
// stands (another tensor type, an argument of another Python type, a failed check, a refused
// launch), and ops.py then runs its own checks, which raise the errors it documents.
// A prefill through ops.py alone is bound by the host: 11.9 us for rope_kv_append, 12.9 for
// varlen_prefill, 9.9 for rms_norm, 10.4 for silu_mul, most of it attribute reads and the
// conversion of up to 26 arguments; through these 3.3, 4.3, 4.6 and 6.3 us (the last with its
// two views).  A 77-token prompt's layer 27.0 -> 12.7 us, now bound by its kernels; four
// 0.5B-sized layers on 2,736 tokens 765 -> 697 us.  Nothing is kept between calls.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdlib>
#include <cstring>

#include "../../include/needle_amd.h"

namespace {

// Entry points of libneedle_amd.so, as ctypes loaded it (init).
decltype(&ndl_rope_kv_append) p_rope_kv_append = nullptr;
decltype(&ndl_varlen_prefill) p_varlen_prefill = nullptr;
decltype(&ndl_rope_varlen_prefill) p_rope_varlen_prefill = nullptr;
decltype(&ndl_varlen_prefill_workspace_bytes) p_prefill_workspace = nullptr;
decltype(&ndl_varlen_prefill_split) p_prefill_split = nullptr;
decltype(&ndl_rms_norm) p_rms_norm = nullptr;
decltype(&ndl_silu_mul) p_silu_mul = nullptr;

// A plain GPU tensor (no subclass, no wrapper of a function transform), or null.
const at::Tensor* gpu_tensor(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || !t.has_storage())
    return nullptr;
  return &t;
}

int dtype_code(at::ScalarType s) {
  switch (s) {
    case at::kBFloat16: return NDL_DTYPE_BF16;
    case at::kHalf: return NDL_DTYPE_F16;
    case at::kFloat: return NDL_DTYPE_F32;
    default: return -1;
  }
}

bool fits_int(int64_t v) { return v >= 0 && v <= 0x7fffffff; }

bool read_int(PyObject* o, int64_t* v) {
  if (!PyLong_CheckExact(o)) return false;
  int over = 0;
  *v = PyLong_AsLongLongAndOverflow(o, &over);
  return over == 0 && fits_int(*v);
}

bool validating() {
  const char* e = std::getenv("NEEDLE_AMD_VALIDATE");
  return e != nullptr && *e != 0 && std::strcmp(e, "0") != 0;
}

ndl_stream_t stream_of(const at::Tensor& t) {
  return (ndl_stream_t)c10::hip::getCurrentHIPStream(t.device().index()).stream();
}

struct Cache {
  int64_t num_blocks, hkv, bs, d;
  int code;
};
bool read_cache(const at::Tensor& c, Cache* r) {
  if (c.dim() != 5 || c.size(0) != 2 || !c.is_contiguous()) return false;
  r->code = dtype_code(c.scalar_type());
  r->num_blocks = c.size(1);
  r->hkv = c.size(2);
  r->bs = c.size(3);
  r->d = c.size(4);
  return r->code >= 0 && fits_int(r->hkv) && fits_int(r->bs) && fits_int(r->d);
}

// Token stride of [T, heads, d] rows of the cache's dtype and device; false if not so.
bool read_rows(const at::Tensor& x, const at::Tensor& cache, int64_t heads, int64_t d,
               int64_t* stride) {
  if (x.dim() != 3 || x.size(1) != heads || x.size(2) != d || x.stride(2) != 1 ||
      x.stride(1) != d || x.device() != cache.device() || x.scalar_type() != cache.scalar_type())
    return false;
  *stride = x.size(0) > 1 ? x.stride(0) : heads * d;
  return true;
}

bool read_int32(const at::Tensor& t, const at::Tensor& cache, int64_t dim) {
  return t.scalar_type() == at::kInt && t.dim() == dim && t.device() == cache.device() &&
         t.stride(dim - 1) == 1;
}

// cos and sin rows [tokens, d], one stride.
bool read_rope(const at::Tensor& cos, const at::Tensor& sin, const at::Tensor& cache,
               int64_t tokens, int64_t d, int64_t* stride) {
  for (const at::Tensor* x : {&cos, &sin})
    if (x->scalar_type() != cache.scalar_type() || x->dim() != 2 || x->size(0) != tokens ||
        x->size(1) != d || x->device() != cache.device() || x->stride(1) != 1)
      return false;
  if (tokens > 1 && cos.stride(0) != sin.stride(0)) return false;
  *stride = tokens > 1 ? cos.stride(0) : d;
  return true;
}

// rope_kv_append(k, v, cos, sin, kv_cache, block_table, context_lens, cu_seqlens): the form
// without q, packed tokens.  True when launched.
PyObject* rope_kv_append(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 8 || p_rope_kv_append == nullptr || validating()) Py_RETURN_NONE;
  const at::Tensor* t[8];
  for (int i = 0; i < 8; ++i)
    if ((t[i] = gpu_tensor(args[i])) == nullptr) Py_RETURN_NONE;
  const at::Tensor &k = *t[0], &v = *t[1], &cos = *t[2], &sin = *t[3], &cache = *t[4],
                   &table = *t[5], &lens = *t[6], &cu = *t[7];
  Cache c;
  int64_t ks, vs, cs;
  if (!read_cache(cache, &c) || c.d % 16 || !read_rows(k, cache, c.hkv, c.d, &ks) ||
      !read_rows(v, cache, c.hkv, c.d, &vs) || !read_int32(table, cache, 2) ||
      !read_int32(lens, cache, 1) || !read_int32(cu, cache, 1))
    Py_RETURN_NONE;
  const int64_t tokens = k.size(0), seqs = table.size(0);
  if (tokens == 0 || v.size(0) != tokens || !read_rope(cos, sin, cache, tokens, c.d, &cs) ||
      lens.size(0) != seqs || cu.size(0) != seqs + 1 || table.size(1) == 0 || !fits_int(seqs) ||
      !fits_int(table.size(1)))
    Py_RETURN_NONE;
  const ndl_stream_t s = stream_of(cache);
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = p_rope_kv_append(nullptr, nullptr, 0, k.data_ptr(), ks, v.data_ptr(), vs, cos.data_ptr(),
                        sin.data_ptr(), cs, cache.data_ptr(), c.num_blocks, (int)c.hkv,
                        (int)c.hkv, (int)c.bs, (int)c.d, c.code, (const int32_t*)table.data_ptr(),
                        table.stride(0), (int)table.size(1), (const int32_t*)cu.data_ptr(),
                        (const int32_t*)lens.data_ptr(), (int)seqs, tokens, s);
  Py_END_ALLOW_THREADS
  if (rc != NDL_OK) Py_RETURN_NONE;
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// varlen_prefill(q, kv_cache, block_table, cu_seqlens, context_lens, max_seqlen, scale,
// num_heads, num_kv_heads, head_dim, max_context_len, cos, sin): the output.
PyObject* varlen_prefill(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 13 || p_varlen_prefill == nullptr || validating()) Py_RETURN_NONE;
  const at::Tensor* t[5];
  for (int i = 0; i < 5; ++i)
    if ((t[i] = gpu_tensor(args[i])) == nullptr) Py_RETURN_NONE;
  const at::Tensor &q = *t[0], &cache = *t[1], &table = *t[2], &cu = *t[3], &lens = *t[4];
  int64_t most, heads, hkv, d, most_ctx, qs, cs = 0;
  if (!read_int(args[5], &most) || !PyFloat_CheckExact(args[6]) || !read_int(args[7], &heads) ||
      !read_int(args[8], &hkv) || !read_int(args[9], &d) || !read_int(args[10], &most_ctx))
    Py_RETURN_NONE;
  const float scale = (float)PyFloat_AS_DOUBLE(args[6]);
  Cache c;
  if (!read_cache(cache, &c) || c.hkv != hkv || c.d != d || !read_rows(q, cache, heads, d, &qs) ||
      !read_int32(table, cache, 2) || !read_int32(cu, cache, 1) || !read_int32(lens, cache, 1))
    Py_RETURN_NONE;
  const int64_t tokens = q.size(0), seqs = table.size(0), width = table.size(1);
  if (tokens == 0 || seqs == 0 || width == 0 || cu.size(0) != seqs + 1 || lens.size(0) != seqs ||
      !fits_int(seqs) || !fits_int(width))
    Py_RETURN_NONE;
  const bool rope = args[11] != Py_None;
  if (rope != (args[12] != Py_None)) Py_RETURN_NONE;
  const void *cosp = nullptr, *sinp = nullptr;
  if (rope) {
    const at::Tensor *cos = gpu_tensor(args[11]), *sin = gpu_tensor(args[12]);
    if (cos == nullptr || sin == nullptr || !read_rope(*cos, *sin, cache, tokens, d, &cs))
      Py_RETURN_NONE;
    cosp = cos->data_ptr();
    sinp = sin->data_ptr();
  }
  at::Tensor out = at::empty({tokens, heads, d}, q.options());
  size_t need = 0;
  // ops.py's rule: the keys of the longest sequence
  const int64_t blocks = c.bs > 0 ? (most_ctx + most + c.bs - 1) / c.bs : 0;
  const int64_t cols = blocks < width ? blocks : width;
  if (cols * c.bs >= NDL_PREFILL_SPLIT_MIN_KEYS)
    need = p_prefill_workspace((int)seqs, tokens, (int)most, (int)cols, (int)heads, (int)hkv,
                               (int)d, (int)c.bs, c.code);
  at::Tensor ws;
  if (need) ws = at::empty({(int64_t)need}, q.options().dtype(at::kByte));
  void* const wsp = need ? ws.data_ptr() : nullptr;
  const ndl_stream_t s = stream_of(cache);
  void* const outp = out.data_ptr();
  const void *qp = q.data_ptr(), *cp = cache.data_ptr();
  const int32_t *tp = (const int32_t*)table.data_ptr(), *cup = (const int32_t*)cu.data_ptr(),
                *lp = (const int32_t*)lens.data_ptr();
  const int64_t bts = table.stride(0);
  int rc;
  Py_BEGIN_ALLOW_THREADS
  if (need)
    rc = p_prefill_split(outp, qp, qs, cosp, sinp, cs, cp, c.num_blocks, tp, bts, (int)width, cup,
                         lp, (int)seqs, tokens, (int)most, (int)most_ctx, (int)heads, (int)hkv,
                         (int)d, (int)c.bs, c.code, scale, wsp, need, s);
  else if (rope)
    rc = p_rope_varlen_prefill(outp, qp, qs, cosp, sinp, cs, cp, c.num_blocks, tp, bts,
                               (int)width, cup, lp, (int)seqs, tokens, (int)most, (int)most_ctx,
                               (int)heads, (int)hkv, (int)d, (int)c.bs, c.code, scale, s);
  else
    rc = p_varlen_prefill(outp, qp, qs, cp, c.num_blocks, tp, bts, (int)width, cup, lp, (int)seqs,
                          tokens, (int)most, (int)most_ctx, (int)heads, (int)hkv, (int)d,
                          (int)c.bs, c.code, scale, s);
  Py_END_ALLOW_THREADS
  if (rc != NDL_OK) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// Row stride of a [rows, width] tensor with contiguous, 16-byte aligned rows like `like`.
bool read_matrix(const at::Tensor& x, const at::Tensor& like, int64_t width, int64_t* stride) {
  if (x.dim() != 2 || x.size(1) != width || x.scalar_type() != like.scalar_type() ||
      x.device() != like.device() || (x.stride(1) != 1 && width != 1))
    return false;
  *stride = x.size(0) > 1 ? x.stride(0) : width;
  return *stride % 8 == 0 && ((uintptr_t)x.data_ptr() & 15u) == 0;
}

// rms_norm(x, weight, eps, residual or None): the norm, or (norm, x + residual).
PyObject* rms_norm(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 4 || p_rms_norm == nullptr || !PyFloat_CheckExact(args[2])) Py_RETURN_NONE;
  const at::Tensor *x = gpu_tensor(args[0]), *w = gpu_tensor(args[1]), *res = nullptr;
  if (x == nullptr || w == nullptr || x->dim() != 2 || x->size(0) == 0) Py_RETURN_NONE;
  const int code = dtype_code(x->scalar_type());
  const int64_t rows = x->size(0), hidden = x->size(1);
  int64_t stride, rstride;
  if (code < 0 || !fits_int(hidden) || !read_matrix(*x, *x, hidden, &stride) || w->dim() != 1 ||
      w->size(0) != hidden || w->scalar_type() != x->scalar_type() || w->device() != x->device() ||
      !w->is_contiguous())
    Py_RETURN_NONE;
  if (args[3] != Py_None) {
    res = gpu_tensor(args[3]);
    if (res == nullptr || !res->is_contiguous() || res->dim() != 2 || res->size(0) != rows ||
        !read_matrix(*res, *x, hidden, &rstride))
      Py_RETURN_NONE;
  }
  at::Tensor out = at::empty({rows, hidden}, x->options()), sum;
  if (res) sum = at::empty({rows, hidden}, x->options());
  const ndl_stream_t s = stream_of(*x);
  void *const outp = out.data_ptr(), *const sump = res ? sum.data_ptr() : nullptr;
  const void *xp = x->data_ptr(), *rp = res ? res->data_ptr() : nullptr, *wp = w->data_ptr();
  const float eps = (float)PyFloat_AS_DOUBLE(args[2]);
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = p_rms_norm(outp, sump, xp, stride, rp, wp, rows, (int)hidden, eps, code, s);
  Py_END_ALLOW_THREADS
  if (rc != NDL_OK) Py_RETURN_NONE;
  if (res == nullptr) return THPVariable_Wrap(std::move(out));
  PyObject* const a = THPVariable_Wrap(std::move(out));
  PyObject* const b = a ? THPVariable_Wrap(std::move(sum)) : nullptr;
  PyObject* const pair = b ? PyTuple_Pack(2, a, b) : nullptr;
  Py_XDECREF(a);
  Py_XDECREF(b);
  return pair;
  END_HANDLE_TH_ERRORS
}

// silu_mul(gate, up): silu(gate) * up.
PyObject* silu_mul(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 2 || p_silu_mul == nullptr) Py_RETURN_NONE;
  const at::Tensor *g = gpu_tensor(args[0]), *u = gpu_tensor(args[1]);
  if (g == nullptr || u == nullptr || g->dim() != 2 || g->size(0) == 0) Py_RETURN_NONE;
  const int code = dtype_code(g->scalar_type());
  const int64_t rows = g->size(0), inter = g->size(1);
  int64_t gs, us;
  if (code < 0 || !fits_int(inter) || !read_matrix(*g, *g, inter, &gs) ||
      !read_matrix(*u, *g, inter, &us) || u->size(0) != rows)
    Py_RETURN_NONE;
  at::Tensor out = at::empty({rows, inter}, g->options());
  const ndl_stream_t s = stream_of(*g);
  void* const outp = out.data_ptr();
  const void *gp = g->data_ptr(), *up = u->data_ptr();
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = p_silu_mul(outp, gp, gs, up, us, rows, (int)inter, code, s);
  Py_END_ALLOW_THREADS
  if (rc != NDL_OK) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// init({name: address}): the entry points to call.
PyObject* init(PyObject*, PyObject* d) {
  auto get = [&](const char* name) -> void* {
    PyObject* const o = PyDict_GetItemString(d, name);
    return o != nullptr && PyLong_Check(o) ? PyLong_AsVoidPtr(o) : nullptr;
  };
  if (!PyDict_Check(d)) {
    PyErr_SetString(PyExc_TypeError, "init takes a dict of addresses");
    return nullptr;
  }
#define NDL_TAKE(var, name) var = (decltype(var))get(name)
  NDL_TAKE(p_rope_kv_append, "ndl_rope_kv_append");
  NDL_TAKE(p_varlen_prefill, "ndl_varlen_prefill");
  NDL_TAKE(p_rope_varlen_prefill, "ndl_rope_varlen_prefill");
  NDL_TAKE(p_prefill_workspace, "ndl_varlen_prefill_workspace_bytes");
  NDL_TAKE(p_prefill_split, "ndl_varlen_prefill_split");
  NDL_TAKE(p_rms_norm, "ndl_rms_norm");
  NDL_TAKE(p_silu_mul, "ndl_silu_mul");
#undef NDL_TAKE
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"init", init, METH_O, nullptr},
    {"rope_kv_append", (PyCFunction)(void (*)(void))rope_kv_append, METH_FASTCALL, nullptr},
    {"varlen_prefill", (PyCFunction)(void (*)(void))varlen_prefill, METH_FASTCALL, nullptr},
    {"rms_norm", (PyCFunction)(void (*)(void))rms_norm, METH_FASTCALL, nullptr},
    {"silu_mul", (PyCFunction)(void (*)(void))silu_mul, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native() {
  PyObject* const m = PyModule_Create(&module);
  // the torch these bindings' inlined code and class layouts are of
  if (m != nullptr && PyModule_AddStringConstant(m, "torch_version", NDL_TORCH_VERSION) != 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
