// direct_calls.cpp - the ops' calls from Python to the kernel library's C ABI, for the forms that a decoder
// layer passes: plain torch.Tensor arguments on one GPU. Each function checks its tensors (type, device,
// shape, strides), then calls the C entry point on torch's current stream and returns its status; for any
// form it does not take, and for anything that does not check out, it returns None before doing anything,
// and the Python wrapper goes its general way, which raises what it always raised. A small call was bound
// by this host work: through Python checks and ctypes a norm took 7.6 us, context attention 14.5 us,
// decode attention 16 us and RoPE with the append 21.9 us of host time.
#include <torch/csrc/autograd/python_variable.h>
#include <torch/version.h>

#include <initializer_list>

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

// A form this file does not take (the Python wrapper handles it).
struct Unhandled {};
void need(bool ok) {
  if (!ok) throw Unhandled{};
}

// A plain tensor (or Parameter) of this type on a GPU; `device` is set by the first and shared by all.
const at::Tensor& tensor(PyObject* o, ScalarType type, int& device) {
  need(THPVariable_CheckExact(o));
  const at::Tensor& t = THPVariable_Unpack(o);
  need(t.defined() && t.is_cuda() && t.layout() == at::kStrided && t.scalar_type() == type && t.numel() > 0);
  if (device < 0) device = t.get_device();
  need(t.get_device() == device);
  return t;
}
const at::Tensor& matrix(PyObject* o, ScalarType type, int& device) {
  const at::Tensor& t = tensor(o, type, device);
  need(t.dim() == 2 && t.stride(1) == 1);
  return t;
}
const at::Tensor& vec(PyObject* o, ScalarType type, int& device) {
  const at::Tensor& t = tensor(o, type, device);
  need(t.dim() == 1 && t.stride(0) == 1);
  return t;
}
// Elements between rows, as the wrappers count them (a single row has no stride of its own).
int64_t row_stride(const at::Tensor& t) { return t.size(0) > 1 ? t.stride(0) : t.size(1); }

double number(PyObject* o) {
  need(PyFloat_CheckExact(o));
  return PyFloat_AS_DOUBLE(o);
}
int64_t integer(PyObject* o) {
  need(PyLong_CheckExact(o));
  const long long v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    throw Unhandled{};
  }
  return v;
}

// An activation scale: a one-element fp32 tensor (read on the device) or a Python float.
struct Scale {
  const float* dev = nullptr;
  float host = 0.f;
};
Scale scale_of(PyObject* o, int& device) {
  if (PyFloat_CheckExact(o)) {
    need(PyFloat_AS_DOUBLE(o) > 0.0);
    return {nullptr, static_cast<float>(PyFloat_AS_DOUBLE(o))};
  }
  const at::Tensor& t = tensor(o, at::kFloat, device);
  need(t.numel() == 1);
  return {static_cast<const float*>(t.data_ptr()), 0.f};
}

uint32_t* error_word(PyObject* o, int& device) {
  return o == Py_None ? nullptr : static_cast<uint32_t*>(tensor(o, at::kInt, device).data_ptr());
}

struct Caches {
  void *k, *v;
  int64_t page_stride, entry_stride, head_stride, pages, page_size, heads, dim;
};
Caches caches_of(PyObject* pair, PyObject* layout, int& device) {
  need(PyTuple_CheckExact(pair) && PyTuple_GET_SIZE(pair) == 2 && PyUnicode_Check(layout));
  const bool nhd = PyUnicode_CompareWithASCIIString(layout, "NHD") == 0;
  need(nhd || PyUnicode_CompareWithASCIIString(layout, "HND") == 0);
  const at::Tensor& k = tensor(PyTuple_GET_ITEM(pair, 0), at::kBFloat16, device);
  const at::Tensor& v = tensor(PyTuple_GET_ITEM(pair, 1), at::kBFloat16, device);
  need(k.dim() == 4 && k.stride(3) == 1 && k.sizes() == v.sizes() && k.strides() == v.strides());
  const int entry = nhd ? 1 : 2, head = nhd ? 2 : 1;
  return {k.data_ptr(), v.data_ptr(), k.stride(0), k.stride(entry), k.stride(head), k.size(0), k.size(entry),
          k.size(head), k.size(3)};
}

// Heads of [nnz, heads * dim] or [nnz, heads, dim].
struct Heads {
  void* p;
  int64_t rows, stride, head_stride, heads;
};
Heads heads_of(PyObject* o, int64_t dim, int& device) {
  const at::Tensor& t = tensor(o, at::kBFloat16, device);
  if (t.dim() == 2) {
    need(t.size(1) % dim == 0 && t.stride(1) == 1);
    return {t.data_ptr(), t.size(0), t.stride(0), dim, t.size(1) / dim};
  }
  need(t.dim() == 3 && t.size(2) == dim && t.stride(2) == 1);
  return {t.data_ptr(), t.size(0), t.stride(0), t.stride(1), t.size(1)};
}

hipStream_t current_stream(int device) {
  PyObject* index = PyLong_FromLong(device);
  PyObject* got = index ? PyObject_CallOneArg(g_raw_stream, index) : nullptr;
  Py_XDECREF(index);
  void* s = got ? PyLong_AsVoidPtr(got) : nullptr;
  Py_XDECREF(got);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    throw Unhandled{};
  }
  return static_cast<hipStream_t>(s);
}

// Runs `body` (which checks, then launches with the GIL released) and maps its outcome.
template <class F>
PyObject* direct(Py_ssize_t got, Py_ssize_t wanted, F&& body) {
  if (got != wanted) Py_RETURN_NONE;
  try {
    return PyLong_FromLong(body());
  } catch (const Unhandled&) {
  } catch (const std::exception&) {  // a tensor without storage and the like: the wrapper reports it
  }
  Py_RETURN_NONE;
}
template <class F>
int launch(F&& f) {
  int st;
  Py_BEGIN_ALLOW_THREADS
  st = f();
  Py_END_ALLOW_THREADS
  return st;
}

// (input, residual, weight, eps)
PyObject* fused_add_rmsnorm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return direct(n, 4, [&] {
    int dev = -1;
    const at::Tensor &x = matrix(a[0], at::kBFloat16, dev), &r = matrix(a[1], at::kBFloat16, dev);
    const at::Tensor& w = vec(a[2], at::kBFloat16, dev);
    const double eps = number(a[3]);
    need(x.sizes() == r.sizes() && w.size(0) == x.size(1) && eps >= 0.0);
    void *xp = x.data_ptr(), *rp = r.data_ptr(), *wp = w.data_ptr();
    const int64_t xs = row_stride(x), rs = row_stride(r), rows = x.size(0), hidden = x.size(1);
    const hipStream_t s = current_stream(dev);
    return launch([&] {
      return g_mas_fused_add_rmsnorm_bf16(static_cast<uint16_t*>(xp), xs, static_cast<uint16_t*>(rp), rs,
                                          static_cast<uint16_t*>(wp), rows, hidden, static_cast<float>(eps), s);
    });
  });
}

// (out, input, residual, weight, scale, eps)
PyObject* fused_add_rmsnorm_quant(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return direct(n, 6, [&] {
    int dev = -1;
    const at::Tensor &x = matrix(a[1], at::kBFloat16, dev), &r = matrix(a[2], at::kBFloat16, dev);
    const at::Tensor& w = vec(a[3], at::kBFloat16, dev);
    const at::Tensor& o = matrix(a[0], at::kFloat8_e4m3fn, dev);
    const Scale q = scale_of(a[4], dev);
    const double eps = number(a[5]);
    need(x.sizes() == r.sizes() && o.sizes() == x.sizes() && w.size(0) == x.size(1) && eps >= 0.0);
    void *op = o.data_ptr(), *xp = x.data_ptr(), *rp = r.data_ptr(), *wp = w.data_ptr();
    const int64_t os = row_stride(o), xs = row_stride(x), rs = row_stride(r), rows = x.size(0), hidden = x.size(1);
    const hipStream_t s = current_stream(dev);
    return launch([&] {
      return g_mas_fused_add_rmsnorm_quant_fp8(static_cast<uint8_t*>(op), os, static_cast<uint16_t*>(xp), xs,
                                               static_cast<uint16_t*>(rp), rs, static_cast<uint16_t*>(wp), q.dev,
                                               q.dev ? 1.0f : q.host, rows, hidden, static_cast<float>(eps), s);
    });
  });
}

// (input, out)
PyObject* silu_and_mul(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return direct(n, 2, [&] {
    int dev = -1;
    const at::Tensor &x = matrix(a[0], at::kBFloat16, dev), &o = matrix(a[1], at::kBFloat16, dev);
    need(x.size(0) == o.size(0) && x.size(1) == 2 * o.size(1));
    void *op = o.data_ptr(), *xp = x.data_ptr();
    const int64_t os = row_stride(o), xs = row_stride(x), rows = x.size(0), inter = o.size(1);
    const hipStream_t s = current_stream(dev);
    return launch([&] {
      return g_mas_silu_and_mul_bf16(static_cast<uint16_t*>(op), os, static_cast<uint16_t*>(xp), xs, rows, inter, s);
    });
  });
}

// (input, out, scale)
PyObject* silu_and_mul_quant(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return direct(n, 3, [&] {
    int dev = -1;
    const at::Tensor &x = matrix(a[0], at::kBFloat16, dev), &o = matrix(a[1], at::kFloat8_e4m3fn, dev);
    const Scale q = scale_of(a[2], dev);
    need(x.size(0) == o.size(0) && x.size(1) == 2 * o.size(1));
    void *op = o.data_ptr(), *xp = x.data_ptr();
    const int64_t os = row_stride(o), xs = row_stride(x), rows = x.size(0), inter = o.size(1);
    const hipStream_t s = current_stream(dev);
    return launch([&] {
      return g_mas_silu_and_mul_quant_fp8(static_cast<uint8_t*>(op), os, static_cast<uint16_t*>(xp), xs, rows, inter,
                                          q.dev, q.dev ? 1.0f : q.host, s);
    });
  });
}

// (positions, query, key, value, head_size, cos_sin_cache, is_neox, batch_indices, paged_kv_cache, kv_indices,
//  kv_indptr, kv_layout, error_flags, q_scale table or None, its interval)
PyObject* rope_append(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return direct(n, 15, [&] {
    int dev = -1;
    const int64_t dim = integer(a[4]);
    need((dim == 32 || dim == 64 || dim == 128 || dim == 256 || dim == 512) && PyBool_Check(a[6]));
    const Heads q = heads_of(a[1], dim, dev), k = heads_of(a[2], dim, dev), v = heads_of(a[3], dim, dev);
    const Caches c = caches_of(a[8], a[11], dev);
    const at::Tensor& cs = matrix(a[5], at::kFloat, dev);
    const at::Tensor &pos = vec(a[0], at::kInt, dev), &batch = vec(a[7], at::kInt, dev);
    const at::Tensor &idx = vec(a[9], at::kInt, dev), &ptr = vec(a[10], at::kInt, dev);
    need(c.dim == dim && cs.size(1) == dim && k.heads == c.heads && v.heads == c.heads);
    need(q.rows == k.rows && q.rows == v.rows && q.rows == pos.size(0) && q.rows == batch.size(0));
    uint32_t* err = error_word(a[12], dev);
    const uint16_t* table = nullptr;
    int64_t table_rows = 0, interval = 0;
    if (a[13] != Py_None) {
      const at::Tensor& t = vec(a[13], at::kBFloat16, dev);
      table = static_cast<const uint16_t*>(t.data_ptr());
      table_rows = t.size(0);
      interval = integer(a[14]);
    }
    const int neox = a[6] == Py_True;
    const auto i32 = [](const at::Tensor& t) { return static_cast<const int32_t*>(t.data_ptr()); };
    const int32_t *pp = i32(pos), *bp = i32(batch), *ip = i32(idx), *rp = i32(ptr);
    const float* cp = static_cast<const float*>(cs.data_ptr());
    const int64_t cstride = cs.stride(0), crows = cs.size(0), nidx = idx.size(0), nbatch = ptr.size(0) - 1;
    const hipStream_t s = current_stream(dev);
    return launch([&] {
      return g_mas_rope_append_paged_kv_cache_bf16(
          static_cast<uint16_t*>(q.p), q.stride, q.head_stride, q.heads, static_cast<uint16_t*>(k.p), k.stride,
          k.head_stride, static_cast<uint16_t*>(v.p), v.stride, v.head_stride, c.heads, pp, cp, cstride, crows, q.rows,
          dim, neox, static_cast<uint16_t*>(c.k), static_cast<uint16_t*>(c.v), c.page_stride, c.entry_stride,
          c.head_stride, c.pages, c.page_size, bp, ip, nidx, rp, nbatch, table, table_rows, interval, err, s);
    });
  });
}

// What the attention calls share: query and out [tokens, heads, dim], int32 block tables and lengths.
struct Attention {
  const at::Tensor *q, *out, *tables, *lens;
  Caches c;
  Scale quant;
  bool fp8;
  uint32_t* err;
};
Attention attention_of(PyObject* query, PyObject* pair, PyObject* tables, PyObject* lens, PyObject* out, PyObject* layout,
                       PyObject* err, PyObject* quant, int& dev) {
  Attention t{};
  t.fp8 = quant != Py_None;
  t.q = &tensor(query, at::kBFloat16, dev);
  t.out = &tensor(out, t.fp8 ? at::kFloat8_e4m3fn : at::kBFloat16, dev);
  t.c = caches_of(pair, layout, dev);
  t.tables = &matrix(tables, at::kInt, dev);
  t.lens = &vec(lens, at::kInt, dev);
  if (t.fp8) t.quant = scale_of(quant, dev);
  t.err = error_word(err, dev);
  need(t.q->dim() == 3 && t.q->size(2) == t.c.dim && t.q->stride(2) == 1 && t.out->sizes() == t.q->sizes() &&
       t.out->stride(2) == 1);
  need(t.q->size(1) % t.c.heads == 0 && (t.c.page_size & (t.c.page_size - 1)) == 0);
  return t;
}

// (query, kv_cache, workspace, block_tables, seq_lens, bmm1_scale, bmm2_scale, out, kv_layout, error_flags,
//  out_quant_scale)
PyObject* decode_attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return direct(n, 11, [&] {
    int dev = -1;
    const Attention t = attention_of(a[0], a[1], a[3], a[4], a[7], a[8], a[9], a[10], dev);
    const at::Tensor& ws = tensor(a[2], at::kByte, dev);
    const double s1 = number(a[5]), s2 = number(a[6]);
    const int64_t batch = t.q->size(0), hq = t.q->size(1), dim = t.c.dim;
    need((dim == 64 || dim == 128 || dim == 256) && hq / t.c.heads <= 16 && t.tables->size(0) >= batch &&
         t.lens->size(0) >= batch);
    void *op = t.out->data_ptr(), *qp = t.q->data_ptr(), *wp = ws.data_ptr();
    const int32_t *tp = static_cast<int32_t*>(t.tables->data_ptr()), *lp = static_cast<int32_t*>(t.lens->data_ptr());
    const int64_t bytes = ws.numel(), os0 = t.out->stride(0), os1 = t.out->stride(1), qs0 = t.q->stride(0),
                  qs1 = t.q->stride(1), ts = t.tables->stride(0), tw = t.tables->size(1);
    const hipStream_t s = current_stream(dev);
    return launch([&] {
      return g_mas_paged_decode_attention_bf16(op, os0, os1, qp, qs0, qs1, t.c.k, t.c.v, t.c.page_stride,
                                               t.c.entry_stride, t.c.head_stride, t.c.pages, t.c.page_size, tp, ts, tw,
                                               lp, batch, hq, t.c.heads, dim, static_cast<float>(s1),
                                               static_cast<float>(s2), t.fp8, t.quant.dev, t.quant.host, wp, bytes,
                                               t.err, s);
    });
  });
}

// (query, kv_cache, workspace or None, block_tables, seq_lens, cum_seq_lens_q, max_q_len, max_kv_len, bmm1_scale,
//  bmm2_scale, out, kv_layout, error_flags, out_quant_scale)
PyObject* context_attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return direct(n, 14, [&] {
    int dev = -1;
    const Attention t = attention_of(a[0], a[1], a[3], a[4], a[10], a[11], a[12], a[13], dev);
    const at::Tensor& cu = vec(a[5], at::kInt, dev);
    void* wp = nullptr;
    int64_t bytes = 0;
    if (a[2] != Py_None) {
      const at::Tensor& ws = tensor(a[2], at::kByte, dev);
      need(ws.is_contiguous());
      wp = ws.data_ptr();
      bytes = ws.numel();
    }
    const int64_t max_q = integer(a[6]), max_kv = integer(a[7]);
    const double s1 = number(a[8]), s2 = number(a[9]);
    const int64_t rows = cu.size(0) - 1, hq = t.q->size(1), dim = t.c.dim;
    need((dim == 64 || dim == 128) && rows >= 0 && t.tables->size(0) >= rows && t.lens->size(0) >= rows);
    void *op = t.out->data_ptr(), *qp = t.q->data_ptr();
    const int32_t *tp = static_cast<int32_t*>(t.tables->data_ptr()), *lp = static_cast<int32_t*>(t.lens->data_ptr()),
                  *cp = static_cast<int32_t*>(cu.data_ptr());
    const int64_t os0 = t.out->stride(0), os1 = t.out->stride(1), qs0 = t.q->stride(0), qs1 = t.q->stride(1),
                  ts = t.tables->stride(0), tw = t.tables->size(1);
    const hipStream_t s = current_stream(dev);
    return launch([&] {
      return g_mas_paged_context_attention_bf16(op, os0, os1, qp, qs0, qs1, t.c.k, t.c.v, t.c.page_stride,
                                                t.c.entry_stride, t.c.head_stride, t.c.pages, t.c.page_size, tp, ts, tw,
                                                lp, cp, rows, max_q, max_kv, hq, t.c.heads, dim,
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
