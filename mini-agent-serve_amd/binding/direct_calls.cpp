// direct_calls.cpp - the ops' calls from Python to the kernel library's C ABI, for the forms that a decoder
// layer passes: plain torch.Tensor arguments on one GPU. Each function checks its tensors (type, device,
// shape, strides), then calls the C entry point on torch's current stream and returns its status; for any
// form it does not take, and for anything that does not check out, it returns None before doing anything,
// and the Python wrapper goes its general way, which raises what it always raised. A small call was bound
// by this host work: through Python checks and ctypes a norm took 7.6 us, context attention 14.5 us,
// decode attention 16 us and RoPE with the append 21.9 us of host time.
#include <torch/csrc/autograd/python_variable.h>
#include <torch/version.h>

#include <exception>

#include "../../include/mas_kernels.h"

namespace {

PyObject* g_raw_stream = nullptr;  // torch._C._cuda_getCurrentRawStream

#define MAS_EACH_FN(F)                    \
  F(mas_fused_add_rmsnorm_bf16)           \
  F(mas_fused_add_rmsnorm_quant_fp8)      \
  F(mas_silu_and_mul_bf16)                \
  F(mas_silu_and_mul_quant_fp8)           \
  F(mas_rope_append_paged_kv_cache_bf16)  \
  F(mas_paged_decode_attention_bf16)      \
  F(mas_paged_context_attention_bf16)
#define MAS_FN(name) decltype(&name) g_##name = nullptr;
MAS_EACH_FN(MAS_FN)
#undef MAS_FN

using at::ScalarType;

// One call's checks: `ok` until an argument is not of a form this file takes (the Python wrapper handles it), and
// the GPU of the first tensor, which all share. The checks after a failed one return nothing to look at, and
// no exception is thrown: unwinding took 2-4 us of every call left to a wrapper.
struct Call {
  bool ok = true;
  int device = -1;

  bool need(bool holds) { return ok = ok && holds; }

  // A plain tensor (or Parameter) of this type on the call's GPU, or null.
  const at::Tensor* tensor(PyObject* o, ScalarType type) {
    if (!need(THPVariable_CheckExact(o))) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!need(t.defined() && t.is_cuda() && t.layout() == at::kStrided && t.scalar_type() == type && t.numel() > 0))
      return nullptr;
    if (device < 0) device = t.get_device();
    return need(t.get_device() == device) ? &t : nullptr;
  }
  const at::Tensor* matrix(PyObject* o, ScalarType type) {
    const at::Tensor* t = tensor(o, type);
    return t != nullptr && need(t->dim() == 2 && t->stride(1) == 1) ? t : nullptr;
  }
  const at::Tensor* vec(PyObject* o, ScalarType type) {
    const at::Tensor* t = tensor(o, type);
    return t != nullptr && need(t->dim() == 1 && t->stride(0) == 1) ? t : nullptr;
  }
  double number(PyObject* o) { return need(PyFloat_CheckExact(o)) ? PyFloat_AS_DOUBLE(o) : 0.0; }
  int64_t integer(PyObject* o) {
    if (!need(PyLong_CheckExact(o))) return 0;
    const long long v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) {
      PyErr_Clear();
      ok = false;
    }
    return v;
  }
};
// Elements between rows, as the wrappers count them (a single row has no stride of its own).
int64_t row_stride(const at::Tensor& t) { return t.size(0) > 1 ? t.stride(0) : t.size(1); }

// An activation scale: a one-element fp32 tensor (read on the device) or a Python float.
struct Scale {
  const float* dev = nullptr;
  float host = 0.f;
};
Scale scale_of(Call& c, PyObject* o) {
  if (PyFloat_CheckExact(o)) {
    c.need(PyFloat_AS_DOUBLE(o) > 0.0);
    return {nullptr, static_cast<float>(PyFloat_AS_DOUBLE(o))};
  }
  const at::Tensor* t = c.tensor(o, at::kFloat);
  return t != nullptr && c.need(t->numel() == 1) ? Scale{static_cast<const float*>(t->data_ptr()), 0.f} : Scale{};
}

uint32_t* error_word(Call& c, PyObject* o) {
  const at::Tensor* t = o == Py_None ? nullptr : c.tensor(o, at::kInt);
  return t != nullptr ? static_cast<uint32_t*>(t->data_ptr()) : nullptr;
}

struct Caches {
  void *k, *v;
  int64_t page_stride, entry_stride, head_stride, pages, page_size, heads, dim;
};
Caches caches_of(Call& c, PyObject* pair, PyObject* layout) {
  if (!c.need(PyTuple_CheckExact(pair) && PyTuple_GET_SIZE(pair) == 2 && PyUnicode_Check(layout))) return {};
  const bool nhd = PyUnicode_CompareWithASCIIString(layout, "NHD") == 0;
  c.need(nhd || PyUnicode_CompareWithASCIIString(layout, "HND") == 0);
  const at::Tensor* k = c.tensor(PyTuple_GET_ITEM(pair, 0), at::kBFloat16);
  const at::Tensor* v = c.tensor(PyTuple_GET_ITEM(pair, 1), at::kBFloat16);
  if (!c.ok || !c.need(k->dim() == 4 && k->stride(3) == 1 && k->sizes() == v->sizes() && k->strides() == v->strides()))
    return {};
  const int entry = nhd ? 1 : 2, head = nhd ? 2 : 1;
  return {k->data_ptr(), v->data_ptr(), k->stride(0), k->stride(entry), k->stride(head), k->size(0), k->size(entry),
          k->size(head), k->size(3)};
}

// Heads of [nnz, heads * dim] or [nnz, heads, dim].
struct Heads {
  void* p;
  int64_t rows, stride, head_stride, heads;
};
Heads heads_of(Call& c, PyObject* o, int64_t dim) {
  const at::Tensor* t = c.tensor(o, at::kBFloat16);
  if (t == nullptr) return {};
  if (t->dim() == 2) {
    if (!c.need(t->size(1) % dim == 0 && t->stride(1) == 1)) return {};
    return {t->data_ptr(), t->size(0), t->stride(0), dim, t->size(1) / dim};
  }
  if (!c.need(t->dim() == 3 && t->size(2) == dim && t->stride(2) == 1)) return {};
  return {t->data_ptr(), t->size(0), t->stride(0), t->stride(1), t->size(1)};
}

hipStream_t current_stream(Call& c) {
  if (!c.ok) return nullptr;
  PyObject* index = PyLong_FromLong(c.device);
  PyObject* got = index ? PyObject_CallOneArg(g_raw_stream, index) : nullptr;
  Py_XDECREF(index);
  void* s = got ? PyLong_AsVoidPtr(got) : nullptr;
  Py_XDECREF(got);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    c.ok = false;
  }
  return static_cast<hipStream_t>(s);
}

// Runs `body`, which checks its arguments with the Call and returns the C entry point's status (its value does not
// count when the checks failed, and nothing was done then).
template <class F>
PyObject* direct(Py_ssize_t got, Py_ssize_t wanted, F&& body) {
  if (got != wanted) Py_RETURN_NONE;
  try {
    Call c;
    const int st = body(c);
    if (c.ok) return PyLong_FromLong(st);
  } catch (const std::exception&) {  // a tensor without storage and the like: the wrapper reports it
  }
  Py_RETURN_NONE;
}
// Calls the C entry point with the GIL released, unless a check failed.
template <class F>
int launch(const Call& c, F&& f) {
  if (!c.ok) return 0;
  int st;
  Py_BEGIN_ALLOW_THREADS
  st = f();
  Py_END_ALLOW_THREADS
  return st;
}

// (input, residual, weight, eps)
PyObject* fused_add_rmsnorm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return direct(n, 4, [&](Call& c) {
    const at::Tensor *x = c.matrix(a[0], at::kBFloat16), *r = c.matrix(a[1], at::kBFloat16);
    const at::Tensor* w = c.vec(a[2], at::kBFloat16);
    const double eps = c.number(a[3]);
    if (!c.ok || !c.need(x->sizes() == r->sizes() && w->size(0) == x->size(1) && eps >= 0.0)) return 0;
    void *xp = x->data_ptr(), *rp = r->data_ptr(), *wp = w->data_ptr();
    const int64_t xs = row_stride(*x), rs = row_stride(*r), rows = x->size(0), hidden = x->size(1);
    const hipStream_t s = current_stream(c);
    return launch(c, [&] {
      return g_mas_fused_add_rmsnorm_bf16(static_cast<uint16_t*>(xp), xs, static_cast<uint16_t*>(rp), rs,
                                          static_cast<uint16_t*>(wp), rows, hidden, static_cast<float>(eps), s);
    });
  });
}

// (out, input, residual, weight, scale, eps)
PyObject* fused_add_rmsnorm_quant(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return direct(n, 6, [&](Call& c) {
    const at::Tensor *x = c.matrix(a[1], at::kBFloat16), *r = c.matrix(a[2], at::kBFloat16);
    const at::Tensor *w = c.vec(a[3], at::kBFloat16), *o = c.matrix(a[0], at::kFloat8_e4m3fn);
    const Scale q = scale_of(c, a[4]);
    const double eps = c.number(a[5]);
    if (!c.ok || !c.need(x->sizes() == r->sizes() && o->sizes() == x->sizes() && w->size(0) == x->size(1) && eps >= 0.0))
      return 0;
    void *op = o->data_ptr(), *xp = x->data_ptr(), *rp = r->data_ptr(), *wp = w->data_ptr();
    const int64_t os = row_stride(*o), xs = row_stride(*x), rs = row_stride(*r), rows = x->size(0), hidden = x->size(1);
    const hipStream_t s = current_stream(c);
    return launch(c, [&] {
      return g_mas_fused_add_rmsnorm_quant_fp8(static_cast<uint8_t*>(op), os, static_cast<uint16_t*>(xp), xs,
                                               static_cast<uint16_t*>(rp), rs, static_cast<uint16_t*>(wp), q.dev,
                                               q.dev ? 1.0f : q.host, rows, hidden, static_cast<float>(eps), s);
    });
  });
}

// (input, out)
PyObject* silu_and_mul(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return direct(n, 2, [&](Call& c) {
    const at::Tensor *x = c.matrix(a[0], at::kBFloat16), *o = c.matrix(a[1], at::kBFloat16);
    if (!c.ok || !c.need(x->size(0) == o->size(0) && x->size(1) == 2 * o->size(1))) return 0;
    void *op = o->data_ptr(), *xp = x->data_ptr();
    const int64_t os = row_stride(*o), xs = row_stride(*x), rows = x->size(0), inter = o->size(1);
    const hipStream_t s = current_stream(c);
    return launch(c, [&] {
      return g_mas_silu_and_mul_bf16(static_cast<uint16_t*>(op), os, static_cast<uint16_t*>(xp), xs, rows, inter, s);
    });
  });
}

// (input, out, scale)
PyObject* silu_and_mul_quant(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return direct(n, 3, [&](Call& c) {
    const at::Tensor *x = c.matrix(a[0], at::kBFloat16), *o = c.matrix(a[1], at::kFloat8_e4m3fn);
    const Scale q = scale_of(c, a[2]);
    if (!c.ok || !c.need(x->size(0) == o->size(0) && x->size(1) == 2 * o->size(1))) return 0;
    void *op = o->data_ptr(), *xp = x->data_ptr();
    const int64_t os = row_stride(*o), xs = row_stride(*x), rows = x->size(0), inter = o->size(1);
    const hipStream_t s = current_stream(c);
    return launch(c, [&] {
      return g_mas_silu_and_mul_quant_fp8(static_cast<uint8_t*>(op), os, static_cast<uint16_t*>(xp), xs, rows, inter,
                                          q.dev, q.dev ? 1.0f : q.host, s);
    });
  });
}

// (positions, query, key, value, head_size, cos_sin_cache, is_neox, batch_indices, paged_kv_cache, kv_indices,
//  kv_indptr, kv_layout, error_flags, q_scale table or None, its interval)
PyObject* rope_append(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return direct(n, 15, [&](Call& c) {
    const int64_t dim = c.integer(a[4]);
    if (!c.need((dim == 32 || dim == 64 || dim == 128 || dim == 256 || dim == 512) && PyBool_Check(a[6]))) return 0;
    const Heads q = heads_of(c, a[1], dim), k = heads_of(c, a[2], dim), v = heads_of(c, a[3], dim);
    const Caches kv = caches_of(c, a[8], a[11]);
    const at::Tensor* cs = c.matrix(a[5], at::kFloat);
    const at::Tensor *pos = c.vec(a[0], at::kInt), *batch = c.vec(a[7], at::kInt);
    const at::Tensor *idx = c.vec(a[9], at::kInt), *ptr = c.vec(a[10], at::kInt);
    uint32_t* err = error_word(c, a[12]);
    if (!c.ok || !c.need(kv.dim == dim && cs->size(1) == dim && k.heads == kv.heads && v.heads == kv.heads &&
                         q.rows == k.rows && q.rows == v.rows && q.rows == pos->size(0) && q.rows == batch->size(0)))
      return 0;
    const uint16_t* table = nullptr;
    int64_t table_rows = 0, interval = 0;
    if (a[13] != Py_None) {
      const at::Tensor* t = c.vec(a[13], at::kBFloat16);
      interval = c.integer(a[14]);
      if (!c.ok) return 0;
      table = static_cast<const uint16_t*>(t->data_ptr());
      table_rows = t->size(0);
    }
    const int neox = a[6] == Py_True;
    const auto i32 = [](const at::Tensor* t) { return static_cast<const int32_t*>(t->data_ptr()); };
    const int32_t *pp = i32(pos), *bp = i32(batch), *ip = i32(idx), *rp = i32(ptr);
    const float* cp = static_cast<const float*>(cs->data_ptr());
    const int64_t cstride = cs->stride(0), crows = cs->size(0), nidx = idx->size(0), nbatch = ptr->size(0) - 1;
    const hipStream_t s = current_stream(c);
    return launch(c, [&] {
      return g_mas_rope_append_paged_kv_cache_bf16(
          static_cast<uint16_t*>(q.p), q.stride, q.head_stride, q.heads, static_cast<uint16_t*>(k.p), k.stride,
          k.head_stride, static_cast<uint16_t*>(v.p), v.stride, v.head_stride, kv.heads, pp, cp, cstride, crows, q.rows,
          dim, neox, static_cast<uint16_t*>(kv.k), static_cast<uint16_t*>(kv.v), kv.page_stride, kv.entry_stride,
          kv.head_stride, kv.pages, kv.page_size, bp, ip, nidx, rp, nbatch, table, table_rows, interval, err, s);
    });
  });
}

// What the attention calls share: query and out [tokens, heads, dim], int32 block tables and lengths.
struct Attention {
  const at::Tensor *q, *out, *tables, *lens;
  Caches kv;
  Scale quant;
  bool fp8;
  uint32_t* err;
};
Attention attention_of(Call& c, PyObject* query, PyObject* pair, PyObject* tables, PyObject* lens, PyObject* out,
                       PyObject* layout, PyObject* err, PyObject* quant) {
  Attention t{};
  t.fp8 = quant != Py_None;
  t.q = c.tensor(query, at::kBFloat16);
  t.out = c.tensor(out, t.fp8 ? at::kFloat8_e4m3fn : at::kBFloat16);
  t.kv = caches_of(c, pair, layout);
  t.tables = c.matrix(tables, at::kInt);
  t.lens = c.vec(lens, at::kInt);
  if (t.fp8) t.quant = scale_of(c, quant);
  t.err = error_word(c, err);
  if (c.ok)
    c.need(t.q->dim() == 3 && t.q->size(2) == t.kv.dim && t.q->stride(2) == 1 && t.out->sizes() == t.q->sizes() &&
           t.out->stride(2) == 1 && t.q->size(1) % t.kv.heads == 0 && (t.kv.page_size & (t.kv.page_size - 1)) == 0);
  return t;
}

// (query, kv_cache, workspace, block_tables, seq_lens, bmm1_scale, bmm2_scale, out, kv_layout, error_flags,
//  out_quant_scale)
PyObject* decode_attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return direct(n, 11, [&](Call& c) {
    const at::Tensor* ws = c.tensor(a[2], at::kByte);
    const double s1 = c.number(a[5]), s2 = c.number(a[6]);
    if (!c.ok) return 0;
    const Attention t = attention_of(c, a[0], a[1], a[3], a[4], a[7], a[8], a[9], a[10]);
    if (!c.ok) return 0;
    const int64_t batch = t.q->size(0), hq = t.q->size(1), dim = t.kv.dim;
    if (!c.need((dim == 64 || dim == 128 || dim == 256) && hq / t.kv.heads <= 16 && t.tables->size(0) >= batch &&
                t.lens->size(0) >= batch))
      return 0;
    void *op = t.out->data_ptr(), *qp = t.q->data_ptr(), *wp = ws->data_ptr();
    const int32_t *tp = static_cast<int32_t*>(t.tables->data_ptr()), *lp = static_cast<int32_t*>(t.lens->data_ptr());
    const int64_t bytes = ws->numel(), os0 = t.out->stride(0), os1 = t.out->stride(1), qs0 = t.q->stride(0),
                  qs1 = t.q->stride(1), ts = t.tables->stride(0), tw = t.tables->size(1);
    const hipStream_t s = current_stream(c);
    return launch(c, [&] {
      return g_mas_paged_decode_attention_bf16(op, os0, os1, qp, qs0, qs1, t.kv.k, t.kv.v, t.kv.page_stride,
                                               t.kv.entry_stride, t.kv.head_stride, t.kv.pages, t.kv.page_size, tp, ts,
                                               tw, lp, batch, hq, t.kv.heads, dim, static_cast<float>(s1),
                                               static_cast<float>(s2), t.fp8, t.quant.dev, t.quant.host, wp, bytes,
                                               t.err, s);
    });
  });
}

// (query, kv_cache, workspace or None, block_tables, seq_lens, cum_seq_lens_q, max_q_len, max_kv_len, bmm1_scale,
//  bmm2_scale, out, kv_layout, error_flags, out_quant_scale)
PyObject* context_attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return direct(n, 14, [&](Call& c) {
    const Attention t = attention_of(c, a[0], a[1], a[3], a[4], a[10], a[11], a[12], a[13]);
    const at::Tensor* cu = c.vec(a[5], at::kInt);
    const at::Tensor* ws = a[2] != Py_None ? c.tensor(a[2], at::kByte) : nullptr;
    const int64_t max_q = c.integer(a[6]), max_kv = c.integer(a[7]);
    const double s1 = c.number(a[8]), s2 = c.number(a[9]);
    if (!c.ok || !c.need(ws == nullptr || ws->is_contiguous())) return 0;
    const int64_t rows = cu->size(0) - 1, hq = t.q->size(1), dim = t.kv.dim;
    if (!c.need((dim == 64 || dim == 128) && rows >= 0 && t.tables->size(0) >= rows && t.lens->size(0) >= rows)) return 0;
    void *op = t.out->data_ptr(), *qp = t.q->data_ptr(), *wp = ws != nullptr ? ws->data_ptr() : nullptr;
    const int64_t bytes = ws != nullptr ? ws->numel() : 0;
    const int32_t *tp = static_cast<int32_t*>(t.tables->data_ptr()), *lp = static_cast<int32_t*>(t.lens->data_ptr()),
                  *cp = static_cast<int32_t*>(cu->data_ptr());
    const int64_t os0 = t.out->stride(0), os1 = t.out->stride(1), qs0 = t.q->stride(0), qs1 = t.q->stride(1),
                  ts = t.tables->stride(0), tw = t.tables->size(1);
    const hipStream_t s = current_stream(c);
    return launch(c, [&] {
      return g_mas_paged_context_attention_bf16(op, os0, os1, qp, qs0, qs1, t.kv.k, t.kv.v, t.kv.page_stride,
                                                t.kv.entry_stride, t.kv.head_stride, t.kv.pages, t.kv.page_size, tp, ts,
                                                tw, lp, cp, rows, max_q, max_kv, hq, t.kv.heads, dim,
                                                static_cast<float>(s1), static_cast<float>(s2), t.fp8, t.quant.dev,
                                                t.quant.host, wp, bytes, t.err, s);
    });
  });
}

// bind(raw_stream, {C entry point's name: its address}): called once, when the kernel library is loaded. Raises,
// with what was bound before still in place, if a name is missing or the library's version is not that of the
// header this file was compiled with, whose signatures it calls.
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 2 || !PyDict_Check(a[1])) {
    PyErr_SetString(PyExc_TypeError, "bind(raw_stream, addresses)");
    return nullptr;
  }
  const auto at_name = [&](const char* name) {
    PyObject* v = PyDict_GetItemString(a[1], name);
    void* p = v ? PyLong_AsVoidPtr(v) : nullptr;
    if (p == nullptr && !PyErr_Occurred()) PyErr_Format(PyExc_KeyError, "%s", name);
    return p;
  };
  void* const version = at_name("mas_version");
#define MAS_FIND(name) void* const p_##name = PyErr_Occurred() ? nullptr : at_name(#name);
  MAS_EACH_FN(MAS_FIND)
#undef MAS_FIND
  if (PyErr_Occurred()) return nullptr;
  if (const int v = reinterpret_cast<decltype(&mas_version)>(version)(); v != MAS_VERSION) {
    PyErr_Format(PyExc_ValueError, "compiled for version %d of the kernel library, loaded with %d", MAS_VERSION, v);
    return nullptr;
  }
#define MAS_SET(name) g_##name = reinterpret_cast<decltype(g_##name)>(p_##name);
  MAS_EACH_FN(MAS_SET)
#undef MAS_SET
  Py_INCREF(a[0]);
  Py_XSETREF(g_raw_stream, a[0]);
  Py_RETURN_NONE;
}

#define MAS_METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {MAS_METHOD(bind),
                         MAS_METHOD(fused_add_rmsnorm),
                         MAS_METHOD(fused_add_rmsnorm_quant),
                         MAS_METHOD(silu_and_mul),
                         MAS_METHOD(silu_and_mul_quant),
                         MAS_METHOD(rope_append),
                         MAS_METHOD(decode_attention),
                         MAS_METHOD(context_attention),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "direct_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_direct_calls() {
  PyObject* m = PyModule_Create(&module);
  // what this file was compiled for: its caller binds it under the same torch and Python only
  if (m != nullptr && (PyModule_AddStringConstant(m, "torch_version", TORCH_VERSION) < 0 ||
                       PyModule_AddIntConstant(m, "python_version", PY_VERSION_HEX >> 16) < 0))
    Py_CLEAR(m);
  return m;
}
