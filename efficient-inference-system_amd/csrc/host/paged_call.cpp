// Native front of the per-layer entry points (CPython extension over ATen): the argument checks,
// the output allocation and the library call of a plain eager call, in one native function each.
// The Python wrappers make ~40 attribute reads on tensors, one allocation and a ctypes call with up
// to 32 converted arguments per call: 6-9 us of host time where the kernels of a small step take
// 4-7 us. Measured (MI355X, host-bound calls back to back): 1 x 8 heads x 64 decode at 128 keys,
// append + prefill of 4 x 256 rows over bf16 pools, q/k/v projections of 333 bf16 rows (see the
// wrappers for the figures).
//
// Every function takes exactly the forms listed in its conditions and returns None for anything
// else (also for tensor subclasses, active function modes and tensors without storage); the Python
// wrapper then does the call itself and raises what is to be raised. Nothing is kept between
// calls except the library's function addresses and the wrappers' workspace dictionary.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>

#include "paged_hip.h"
#include "pa_internal.h"

namespace {

struct Lib {
  decltype(&pa_decode) decode = nullptr;
  decltype(&pa_decode_workspace_size) decode_ws = nullptr;
  decltype(&pa_prefill) prefill = nullptr;
  decltype(&paged_internal_prefill_workspace) prefill_ws = nullptr;
  decltype(&pa_kv_append) append = nullptr;
  decltype(&pa_linear_rows) linear = nullptr;
  decltype(&pa_qkv_append) qkv = nullptr;
};
Lib L;
bool ready = false;
PyObject* workspaces = nullptr;  // {(device index, kind): uint8 tensor}
PyObject* raw_stream = nullptr;  // torch._C._cuda_getCurrentRawStream
PyObject* fail = nullptr;        // _lib.check(status, what)
PyObject* side_workspace = nullptr;  // _call_workspace(device, bytes, kind): off the default stream
PyObject* splits = nullptr;      // default_split_blocks(batch, heads, max_pages, device, ordered)
PyObject *kind_decode, *kind_prefill, *kind_balanced, *str_device;

using Tensor = at::Tensor;

// The plain tensor behind o, or null.
const Tensor* plain(PyObject* o) {
  return THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr;
}
bool optional(PyObject* o, const Tensor*& t) {
  t = nullptr;
  return o == Py_None || (t = plain(o)) != nullptr;
}
bool on_gpu(const Tensor* t) { return t != nullptr && t->is_cuda(); }
// An optional operand that a kernel reads: on the GPU, whole, of at least `entries` elements.
bool readable(const Tensor* t, int64_t entries) {
  return t == nullptr || (t->is_cuda() && t->is_contiguous() && t->numel() >= entries);
}
int dtype_of(const Tensor& t) {
  return t.scalar_type() == at::kFloat ? PA_DTYPE_F32 : (t.scalar_type() == at::kBFloat16 ? PA_DTYPE_BF16 : -1);
}
bool i32(const Tensor* t) { return on_gpu(t) && t->scalar_type() == at::kInt && t->is_contiguous(); }
bool pools(const Tensor* k, const Tensor* v) {
  return on_gpu(k) && on_gpu(v) && k->dim() == 4 && k->sizes() == v->sizes() && k->scalar_type() == v->scalar_type() &&
         k->is_contiguous() && v->is_contiguous() && dtype_of(*k) >= 0;
}
bool fits32(int64_t n) { return n >= 0 && n <= 0x7fffffff; }
const void* data(const Tensor* t) { return t ? t->data_ptr() : nullptr; }

bool stream_of(const Tensor& t, void*& stream) {
  PyObject* idx = PyLong_FromLong(t.get_device());
  PyObject* s = idx ? PyObject_CallOneArg(raw_stream, idx) : nullptr;
  Py_XDECREF(idx);
  if (s == nullptr) return false;
  stream = PyLong_AsVoidPtr(s);
  Py_DECREF(s);
  return !PyErr_Occurred();
}

// The workspace of a call on tensor t (of Python object o): the default stream's kept one if it holds
// `bytes` (null: the wrapper allocates), on another stream that stream's, a reference to it in `ref`.
struct Ref {
  PyObject* o = nullptr;
  ~Ref() { Py_XDECREF(o); }
};
void* workspace(PyObject* o, const Tensor& t, void* stream, PyObject* kind, size_t bytes, Ref& ref) {
  if (stream != nullptr) {
    PyObject* dev = PyObject_GetAttr(o, str_device);
    ref.o = dev ? PyObject_CallFunction(side_workspace, "OnO", dev, (Py_ssize_t)bytes, kind) : nullptr;
    Py_XDECREF(dev);
    const Tensor* ws = ref.o ? plain(ref.o) : nullptr;
    return ws ? ws->data_ptr() : nullptr;
  }
  PyObject* idx = PyLong_FromLong(t.get_device());
  PyObject* key = idx ? PyTuple_Pack(2, idx, kind) : nullptr;
  PyObject* w = key ? PyDict_GetItemWithError(workspaces, key) : nullptr;
  Py_XDECREF(idx);
  Py_XDECREF(key);
  const Tensor* ws = w ? plain(w) : nullptr;
  return ws != nullptr && (size_t)ws->numel() >= bytes ? ws->data_ptr() : nullptr;
}

// New reference to `out` wrapped (or to the given object) after a successful status; otherwise the
// exception that _lib.check raises.
PyObject* finish(int status, const char* what, PyObject* given, const Tensor& out) {
  if (status != PA_OK) {
    PyObject* r = PyObject_CallFunction(fail, "is", status, what);
    Py_XDECREF(r);
    return nullptr;
  }
  if (given != nullptr && given != Py_None) {
    Py_INCREF(given);
    return given;
  }
  return THPVariable_Wrap(out);
}

// The library call without the GIL, as ctypes makes it. (An argument may throw: the GIL comes back
// on every way out.)
template <typename F>
int unlocked(F&& f) {
  struct Gil {
    PyThreadState* ts = PyEval_SaveThread();
    ~Gil() { PyEval_RestoreThread(ts); }
  } gil;
  return f();
}

bool usable(Py_ssize_t n, Py_ssize_t want) {
  return ready && n == want && !at::impl::torch_function_mode_enabled();
}

// A body that returns null without a Python error set (a form left to the wrapper) gives None, and so
// does one that throws: the wrapper repeats the call and meets the same error with its own message.
template <typename F>
PyObject* guarded(F&& body) {
  try {
    PyObject* r = body();
    if (r == nullptr && !PyErr_Occurred()) Py_RETURN_NONE;
    return r;
  } catch (const std::exception&) {
    if (PyErr_Occurred()) PyErr_Clear();
    Py_RETURN_NONE;
  }
}

// What decode and prefill share: q, pools, page table, lengths and out in the plain forms.
struct Attn {
  const Tensor *q, *k, *v, *pt, *sl, *cl, *out;
  Tensor made;
  int64_t B, H, T, Hd, nblk, bs, pages, pt_stride, split;
  bool parse(PyObject* const* a, PyObject* split_o, PyObject* out_o) {
    q = plain(a[0]); k = plain(a[1]); v = plain(a[2]); pt = plain(a[3]); sl = plain(a[4]); cl = plain(a[5]);
    if (!on_gpu(q) || !pools(k, v) || !i32(pt) || !i32(sl) || !i32(cl) || !optional(out_o, out)) return false;
    if (q->dim() != 4 || dtype_of(*q) < 0 || q->stride(3) != 1 || pt->dim() != 2) return false;
    B = q->size(0); H = q->size(1); T = q->size(2); Hd = q->size(3);
    nblk = k->size(0); bs = k->size(2);
    pages = pt->size(1); pt_stride = pt->stride(0);
    if (k->size(1) != H || k->size(3) != Hd || B == 0 || pages == 0) return false;
    if (pt->size(0) < B || sl->numel() < B || cl->numel() < B) return false;
    if (!fits32(B) || !fits32(H) || !fits32(T) || !fits32(Hd) || !fits32(bs) || !fits32(pages)) return false;
    if (out != nullptr && (!out->is_cuda() || out->device() != q->device() || out->sizes() != q->sizes() ||
                           out->scalar_type() != q->scalar_type() || out->stride(3) != 1))
      return false;
    split = 0;
    if (split_o != Py_None) {
      split = PyLong_Check(split_o) ? PyLong_AsLongLong(split_o) : -(1LL << 40);
      if (PyErr_Occurred()) PyErr_Clear();
      if (split < -0x7fffffff || split > 0x7fffffff) return false;
    }
    return true;
  }
  const Tensor& result() {
    if (out != nullptr) return *out;
    made = at::empty_like(*q);
    return made;
  }
};

// decode(q, k_pool, v_pool, page_table, seq_lens, current_lengths, order, split_blocks, out)
PyObject* decode(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!usable(n, 9)) Py_RETURN_NONE;
  return guarded([&]() -> PyObject* {
    Attn t;
    const Tensor* order;
    if (!t.parse(a, a[7], a[8]) || t.T != 1 || !optional(a[6], order)) return nullptr;
    if (order != nullptr && !(order->scalar_type() == at::kInt && readable(order, t.B))) return nullptr;
    if (a[7] == Py_None) {
      PyObject* dev = PyObject_GetAttr(a[0], str_device);
      PyObject* sb = dev ? PyObject_CallFunction(splits, "LLLOO", (long long)t.B, (long long)t.H, (long long)t.pages,
                                                 dev, order ? Py_True : Py_False)
                         : nullptr;
      Py_XDECREF(dev);
      if (sb == nullptr) return nullptr;
      t.split = PyLong_AsLongLong(sb);
      Py_DECREF(sb);
      if (PyErr_Occurred()) return nullptr;
    }
    const size_t need = t.bs == 16 ? L.decode_ws(t.B, t.H, t.Hd, t.pages, t.split) : 0;
    void* stream;
    if (!stream_of(*t.q, stream)) return nullptr;
    Ref held;
    void* ws = need ? workspace(a[0], *t.q, stream, t.split < 0 ? kind_balanced : kind_decode, need, held) : nullptr;
    if (need && ws == nullptr) return nullptr;
    const Tensor& o = t.result();
    const void* ord = data(order);
    const int st = unlocked([&] {
      return L.decode(t.q->data_ptr(), t.q->stride(0), t.q->stride(1), o.data_ptr(), o.stride(0), o.stride(1),
                      dtype_of(*t.q), t.k->data_ptr(), t.v->data_ptr(), dtype_of(*t.k), t.nblk,
                      t.pt->data_ptr<int>(), t.pt_stride, t.pages, t.sl->data_ptr<int>(), t.cl->data_ptr<int>(),
                      static_cast<const int32_t*>(ord), t.B, t.H, t.Hd, t.bs, (float)(1.0 / std::sqrt((double)t.Hd)),
                      t.split, ws, need, stream);
    });
    return finish(st, "pa_decode", a[8], o);
  });
}

// prefill(q, k_pool, v_pool, page_table, seq_lens, current_lengths, split_blocks, out)
PyObject* prefill(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!usable(n, 8)) Py_RETURN_NONE;
  return guarded([&]() -> PyObject* {
    Attn t;
    if (a[6] == Py_None || !t.parse(a, a[6], a[7])) return nullptr;
    const size_t need = t.bs == 16 ? L.prefill_ws(dtype_of(*t.k), t.B, t.H, t.T, t.Hd, t.pages, t.split) : 0;
    void* stream;
    if (!stream_of(*t.q, stream)) return nullptr;
    Ref held;
    void* ws = need ? workspace(a[0], *t.q, stream, kind_prefill, need, held) : nullptr;
    if (need && ws == nullptr) return nullptr;
    const Tensor& o = t.result();
    const int st = unlocked([&] {
      return L.prefill(t.q->data_ptr(), t.q->stride(0), t.q->stride(1), t.q->stride(2), o.data_ptr(), o.stride(0),
                       o.stride(1), o.stride(2), dtype_of(*t.q), t.k->data_ptr(), t.v->data_ptr(), dtype_of(*t.k),
                       t.nblk, t.pt->data_ptr<int>(), t.pt_stride, t.pages, t.sl->data_ptr<int>(),
                       t.cl->data_ptr<int>(), t.B, t.H, t.T, t.Hd, t.bs, (float)(1.0 / std::sqrt((double)t.Hd)),
                       t.split, ws, need, stream);
    });
    return finish(st, "pa_prefill", a[7], o);
  });
}

// kv_append(k_new, v_new, k_pool, v_pool, slot_mapping): True, or None
PyObject* kv_append(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!usable(n, 5)) Py_RETURN_NONE;
  return guarded([&]() -> PyObject* {
    const Tensor *kn = plain(a[0]), *vn = plain(a[1]), *k = plain(a[2]), *v = plain(a[3]), *sm = plain(a[4]);
    if (!on_gpu(kn) || !on_gpu(vn) || !pools(k, v) || !i32(sm) || kn->dim() != 4 || kn->sizes() != vn->sizes() ||
        kn->scalar_type() != vn->scalar_type() || kn->strides() != vn->strides() || kn->stride(3) != 1 ||
        dtype_of(*kn) < 0)
      return nullptr;
    const int64_t B = kn->size(0), H = kn->size(1), T = kn->size(2), Hd = kn->size(3);
    if (sm->numel() != B * T || k->size(1) != H || k->size(3) != Hd || !fits32(B) || !fits32(H) || !fits32(T) ||
        !fits32(Hd) || !fits32(k->size(2)))
      return nullptr;
    void* stream;
    if (!stream_of(*kn, stream)) return nullptr;
    const int st = unlocked([&] {
      return L.append(kn->data_ptr(), vn->data_ptr(), kn->stride(0), kn->stride(1), kn->stride(2), dtype_of(*kn),
                      k->data_ptr(), v->data_ptr(), dtype_of(*k), k->size(0), sm->data_ptr<int>(), B, H, T, Hd,
                      k->size(2), stream);
    });
    return finish(st, "pa_kv_append", Py_True, *kn);
  });
}

// A [rows, features] GPU tensor of dtype dt (-1: either) with unit column stride.
bool rows2d(const Tensor* t, int dt) {
  return on_gpu(t) && t->dim() == 2 && t->stride(1) == 1 && dtype_of(*t) >= 0 && (dt < 0 || dtype_of(*t) == dt);
}
bool typed(const Tensor* t, int dt) { return t == nullptr || dtype_of(*t) == dt; }
bool holds(const Tensor* t, int64_t rows, int64_t cols) { return t == nullptr || (t->size(0) >= rows && t->size(1) >= cols); }
// A layer's parameters: weight [rows, cols], bias.
bool parameters(const Tensor* w, const Tensor* b, int64_t rows, int64_t cols) {
  return w->dim() == 2 && w->size(0) == rows && w->size(1) == cols && readable(w, rows * cols) && readable(b, rows);
}

// linear_rows(x, weight, bias, ln_weight, ln_bias, ln_eps, gelu, residual, out, copy_to)
PyObject* linear_rows(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!usable(n, 10)) Py_RETURN_NONE;
  return guarded([&]() -> PyObject* {
    const Tensor *x = plain(a[0]), *w = plain(a[1]), *b, *lw, *lb, *res, *out, *cp;
    if (!rows2d(x, -1) || w == nullptr || !optional(a[2], b) || !optional(a[3], lw) || !optional(a[4], lb) ||
        !optional(a[7], res) || !optional(a[8], out) || !optional(a[9], cp))
      return nullptr;
    const int dt = dtype_of(*x);
    const int64_t M = x->size(0), K = x->size(1);
    if (w->dim() != 2 || w->size(1) != K || !typed(w, dt) || !typed(b, dt) || !typed(lw, dt) || !typed(lb, dt))
      return nullptr;
    const int64_t N = w->size(0);
    if ((res && !rows2d(res, dt)) || (out && !rows2d(out, dt)) || (cp && !rows2d(cp, dt))) return nullptr;
    if (!parameters(w, b, N, K) || !readable(lw, K) || !readable(lb, K)) return nullptr;
    if (!holds(res, M, N) || !holds(out, M, N) || !holds(cp, M, N)) return nullptr;
    if (!fits32(M) || !fits32(K) || !fits32(N)) return nullptr;
    const double eps = PyFloat_AsDouble(a[5]);
    const int gelu = PyObject_IsTrue(a[6]);
    void* stream;
    if (PyErr_Occurred() || !stream_of(*x, stream)) return nullptr;
    const Tensor made = out ? Tensor() : at::empty({M, N}, x->options());
    const Tensor& o = out ? *out : made;
    const int st = unlocked([&] {
      return L.linear(x->data_ptr(), x->stride(0), M, K, w->data_ptr(), data(b), N, data(lw), data(lb), (float)eps,
                      gelu, data(res), res ? res->stride(0) : 0, o.data_ptr(), o.stride(0),
                      const_cast<void*>(data(cp)), cp ? cp->stride(0) : 0, dt, stream);
    });
    return finish(st, "pa_linear_rows", a[8], o);
  });
}

// qkv_append(x, ln_weight, ln_bias, ln_eps, wq, bq, wk, bk, wv, bv, k_pool, v_pool, slot_mapping, out)
PyObject* qkv_append(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!usable(n, 14)) Py_RETURN_NONE;
  return guarded([&]() -> PyObject* {
    const Tensor *x = plain(a[0]), *lw, *lb, *w[3], *b[3], *k = plain(a[10]), *v = plain(a[11]), *sm = plain(a[12]), *out;
    if (!rows2d(x, -1) || !optional(a[1], lw) || !optional(a[2], lb) || !optional(a[13], out)) return nullptr;
    const int dt = dtype_of(*x);
    if (!typed(lw, dt) || !typed(lb, dt)) return nullptr;
    for (int i = 0; i < 3; ++i) {
      w[i] = plain(a[4 + 2 * i]);
      if (w[i] == nullptr || !optional(a[5 + 2 * i], b[i]) || !typed(w[i], dt) || !typed(b[i], dt)) return nullptr;
    }
    const int64_t M = x->size(0), D = x->size(1);
    for (int i = 0; i < 3; ++i)
      if (!parameters(w[i], b[i], D, D)) return nullptr;
    if (!readable(lw, D) || !readable(lb, D)) return nullptr;
    if ((out && (!rows2d(out, dt) || !holds(out, M, D))) || !pools(k, v) || sm == nullptr || sm->scalar_type() != at::kInt ||
        !readable(sm, M) || !fits32(M) || !fits32(D) || !fits32(k->size(1)) ||
        !fits32(k->size(2)) || !fits32(k->size(3)))
      return nullptr;
    const double eps = PyFloat_AsDouble(a[3]);
    void* stream;
    if (PyErr_Occurred() || !stream_of(*x, stream)) return nullptr;
    const Tensor made = out ? Tensor() : at::empty({M, D}, x->options());
    const Tensor& o = out ? *out : made;
    const int st = unlocked([&] {
      return L.qkv(x->data_ptr(), x->stride(0), M, D, data(lw), data(lb), (float)eps, w[0]->data_ptr(), data(b[0]),
                   w[1]->data_ptr(), data(b[1]), w[2]->data_ptr(), data(b[2]), o.data_ptr(), o.stride(0),
                   k->data_ptr(), v->data_ptr(), dtype_of(*k), k->size(0), static_cast<const int32_t*>(sm->data_ptr()),
                   k->size(1), k->size(3), k->size(2), dt, stream);
    });
    return finish(st, "pa_qkv_append", a[13], o);
  });
}

// bind({name: address}, workspaces, raw stream lookup, check, default_split_blocks, _call_workspace): the
// functions serve calls from here on.
PyObject* bind(PyObject*, PyObject* args) {
  PyObject *addr, *ws, *rs, *ck, *sp, *sw;
  if (!PyArg_ParseTuple(args, "O!O!OOOO", &PyDict_Type, &addr, &PyDict_Type, &ws, &rs, &ck, &sp, &sw)) return nullptr;
  auto get = [&](const char* name, auto& fn) {
    PyObject* o = PyDict_GetItemString(addr, name);
    if (o == nullptr) {
      PyErr_Format(PyExc_KeyError, "no address for %s", name);
      return false;
    }
    fn = reinterpret_cast<std::remove_reference_t<decltype(fn)>>(PyLong_AsVoidPtr(o));
    return !PyErr_Occurred();
  };
  if (!get("pa_decode", L.decode) || !get("pa_decode_workspace_size", L.decode_ws) ||
      !get("pa_prefill", L.prefill) ||
      !get("paged_internal_prefill_workspace", L.prefill_ws) || !get("pa_kv_append", L.append) ||
      !get("pa_linear_rows", L.linear) || !get("pa_qkv_append", L.qkv))
    return nullptr;
  Py_INCREF(ws); Py_INCREF(rs); Py_INCREF(ck); Py_INCREF(sp); Py_INCREF(sw);
  Py_XSETREF(workspaces, ws);
  Py_XSETREF(raw_stream, rs);
  Py_XSETREF(fail, ck);
  Py_XSETREF(splits, sp);
  Py_XSETREF(side_workspace, sw);
  ready = true;
  Py_RETURN_NONE;
}

PyCFunction fast(PyObject* (*f)(PyObject*, PyObject* const*, Py_ssize_t)) {
  return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f));
}

PyMethodDef methods[] = {
    {"bind", bind, METH_VARARGS, "Give the library's function addresses."},
    {"decode", fast(decode), METH_FASTCALL, "Decode attention of a plain call, or None."},
    {"prefill", fast(prefill), METH_FASTCALL, "Prefill attention of a plain call, or None."},
    {"kv_append", fast(kv_append), METH_FASTCALL, "KV append of a plain call, or None."},
    {"linear_rows", fast(linear_rows), METH_FASTCALL, "Linear layer over a step's rows of a plain call, or None."},
    {"qkv_append", fast(qkv_append), METH_FASTCALL, "q/k/v projections and append of a plain call, or None."},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_paged_call", "Native front of the per-layer entry points.", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__paged_call(void) {
  kind_decode = PyUnicode_InternFromString("decode");
  kind_prefill = PyUnicode_InternFromString("prefill");
  kind_balanced = PyUnicode_InternFromString("balanced");
  str_device = PyUnicode_InternFromString("device");
  return kind_decode && kind_prefill && kind_balanced && str_device ? PyModule_Create(&module) : nullptr;
}
