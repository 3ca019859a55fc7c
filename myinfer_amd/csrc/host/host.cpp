// The host path of one attention layer's step, over torch tensors: the checks, the descriptors, the output
// and the foreign call of kernels.prepare_attention and AppendCall for the forms a model's layers use, and
// the views QuantizedKVCache.fetch returns.
//
// In Python the two calls of a decode step cost about 45 us of host time, three times their kernels' time
// on a 4096-token cache of 8 heads; here about 10. Every function returns None for anything but those
// forms (other types, devices, strides, a call the library refuses): the Python path then serves the call
// or raises, so that what is accepted and what is refused has one definition. A launch that failed is not
// tried again: the Python side gets its (negative) status to raise. The interpreter lock is released
// around the library's calls, which may wait for room in a full queue.

#include <ATen/ATen.h>
#include <string.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/version.h>

#include "../../../include/kvq.h"

namespace {

using AttnFn = int (*)(const kvq_rows*, const kvq_qtensor*, const kvq_qtensor*, const int32_t*, const kvq_rows*, int, int,
                       int, int, int, int, int, int, int, float, int, int, void*, size_t, void*);
using SizeFn = size_t (*)(int, int, int, int, int, int, int);
using AppendFn = int (*)(const kvq_rows*, const kvq_qtensor*, const kvq_rows*, const kvq_qtensor*, int64_t, int, int, int,
                         int, int, int, int, void*);
using RopeAppendFn = int (*)(const kvq_rows*, const kvq_qtensor*, const kvq_rows*, const kvq_qtensor*,
                             const kvq_rope_params*, int64_t, int, int, int, int, int, int, int, void*);

struct {
  AttnFn decode = nullptr, prefill = nullptr;
  SizeFn decode_ws = nullptr, prefill_ws = nullptr;
} g;

// The destination of an AppendCall (myinfer_amd/_lib.py, AppendState).
struct AppendState {
  void* fn;
  const kvq_qtensor *kq, *vq;
  const kvq_rope_params* rope;  // or NULL
  int64_t B, H, rows, code_words, groups;
  int32_t bits, group, code, device;
  void* stream;
};

PyObject* none() { Py_RETURN_NONE; }

// What a library call that did not return KVQ_OK becomes: see above. (Nothing was launched by a refused one.)
PyObject* failed(int rc) {
  if (rc == KVQ_ERR_HIP) return PyLong_FromLong(rc);
  return none();
}

// Releases the interpreter lock while it lives.
struct Unlocked {
  PyThreadState* st = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(st); }
};

int dtype_code(at::ScalarType t) {
  return t == at::kHalf ? KVQ_DTYPE_F16 : t == at::kBFloat16 ? KVQ_DTYPE_BF16 : -1;
}

// Rows that the kernels read in place: 4-D, unit stride along D, 16-byte aligned, strides of 8 elements.
bool rows_of(const at::Tensor& t, kvq_rows* r) {
  if (t.dim() != 4 || t.stride(3) != 1) return false;
  *r = {t.data_ptr(), t.stride(0), t.stride(1), t.stride(2)};
  return !(((uintptr_t)r->data | 2 * (uintptr_t)(r->stride_b | r->stride_h | r->stride_l)) % 16);
}

struct Triple {
  at::Tensor c, s, b;
};
bool triple_of(PyObject* o, Triple* t) {
  if (!PyTuple_Check(o) || PyTuple_GET_SIZE(o) != 3) return false;
  PyObject* const* x = &PyTuple_GET_ITEM(o, 0);
  if (!THPVariable_Check(x[0]) || !THPVariable_Check(x[1]) || !THPVariable_Check(x[2])) return false;
  t->c = THPVariable_Unpack(x[0]);
  t->s = THPVariable_Unpack(x[1]);
  t->b = THPVariable_Unpack(x[2]);
  return true;
}
bool qtensor_of(const Triple& t, int64_t B, int64_t Hkv, int64_t S, int64_t D, int bits, int group, at::ScalarType dt,
                const at::Device& dev, int32_t* range_exp, kvq_qtensor* q) {
  const auto& c = t.c;
  if (c.dim() != 4 || t.s.dim() != 4 || t.b.dim() != 4) return false;
  if ((c.scalar_type() != at::kUInt32 && c.scalar_type() != at::kInt) || t.s.scalar_type() != dt ||
      t.b.scalar_type() != dt)
    return false;
  if (c.device() != dev || t.s.device() != dev || t.b.device() != dev) return false;
  if (c.size(0) != B || c.size(1) != Hkv || c.size(2) != S || c.size(3) * 32 != D * bits) return false;
  if (t.s.size(0) != B || t.s.size(1) != Hkv || t.s.size(2) != S || t.s.size(3) * group != D) return false;
  if (t.s.sizes() != t.b.sizes() || t.s.strides() != t.b.strides()) return false;
  if (c.stride(3) != 1 || t.s.stride(3) != 1) return false;
  *q = {(uint32_t*)c.data_ptr(), t.s.data_ptr(), t.b.data_ptr(), c.stride(0), c.stride(1), c.stride(2),
        t.s.stride(0), t.s.stride(1), t.s.stride(2), range_exp};
  return true;
}

// attention(queries, keys, values, scale, causal, window, seq_lens, group_size, bits, prefill, k_range, v_range,
//           workspace, stream) -> the output, the workspace bytes needed if the given ones are too few, the negative
//           status of a failed launch, or None
PyObject* attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 14 || !g.decode || !THPVariable_Check(a[0])) return none();
  try {
    const at::Tensor& q = THPVariable_Unpack(a[0]);
    Triple k, v;
    if (!triple_of(a[1], &k) || !triple_of(a[2], &v)) return none();
    const double scale = PyFloat_AsDouble(a[3]);
    const long causal = PyLong_AsLong(a[4]), window = PyLong_AsLong(a[5]);
    const long group = PyLong_AsLong(a[7]), bits = PyLong_AsLong(a[8]), prefill = PyLong_AsLong(a[9]);
    void* kw = PyLong_AsVoidPtr(a[10]);
    void* vw = PyLong_AsVoidPtr(a[11]);
    void* stream = PyLong_AsVoidPtr(a[13]);
    if (PyErr_Occurred()) {
      PyErr_Clear();
      return none();
    }
    kvq_rows qr;
    const int code = dtype_code(q.scalar_type());
    if (code < 0 || !q.is_cuda() || !rows_of(q, &qr) || (bits != 4 && bits != 8) || group <= 0 || window < 0) return none();
    const int64_t B = q.size(0), Hq = q.size(1), L = q.size(2), D = q.size(3);
    if (k.c.dim() != 4) return none();
    const int64_t Hkv = k.c.size(1), S = k.c.size(2);
    if (B <= 0 || Hkv <= 0 || L <= 0 || S <= 0 || Hq % Hkv || Hq <= 0) return none();
    if (B > INT32_MAX || Hq > INT32_MAX || L > INT32_MAX || S > INT32_MAX || window > INT32_MAX) return none();
    kvq_qtensor kq, vq;
    const at::Device dev = q.device();
    if (!qtensor_of(k, B, Hkv, S, D, bits, group, q.scalar_type(), dev, (int32_t*)kw, &kq) ||
        !qtensor_of(v, B, Hkv, S, D, bits, group, q.scalar_type(), dev, (int32_t*)vw, &vq))
      return none();
    const int32_t* lens = nullptr;
    if (a[6] != Py_None) {
      if (!THPVariable_Check(a[6])) return none();
      const at::Tensor& t = THPVariable_Unpack(a[6]);
      if (t.scalar_type() != at::kInt || t.device() != dev || t.numel() != B || !t.is_contiguous()) return none();
      lens = (const int32_t*)t.data_ptr();
    }
    const size_t need = (prefill ? g.prefill_ws : g.decode_ws)((int)B, (int)Hq, (int)Hkv, (int)L, (int)D, (int)S, (int)window);
    if (need == 0) return none();
    if (!THPVariable_Check(a[12])) return PyLong_FromSize_t(need);
    const at::Tensor& ws = THPVariable_Unpack(a[12]);
    if (ws.nbytes() < need) return PyLong_FromSize_t(need);
    at::Tensor out = at::empty({B, Hq, L, D}, q.options().requires_grad(false));
    const kvq_rows orr = {out.data_ptr(), Hq * L * D, L * D, D};
    void* const wp = ws.data_ptr();
    const size_t wn = ws.nbytes();
    int rc;
    {
      Unlocked u;
      rc = (prefill ? g.prefill : g.decode)(&qr, &kq, &vq, lens, &orr, (int)B, (int)Hq, (int)Hkv, (int)L, (int)D, (int)S,
                                            (int)bits, (int)group, code, (float)scale, (int)causal, (int)window, wp, wn,
                                            stream);
    }
    if (rc != KVQ_OK) return failed(rc);
    return THPVariable_Wrap(std::move(out));
  } catch (...) {
    return none();
  }
}

// append(state address, keys, values, row_offset, rope_offset) -> True, the negative status of a failed launch, or None
PyObject* append(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 5 || !THPVariable_Check(a[1]) || !THPVariable_Check(a[2])) return none();
  try {
    const AppendState* st = (const AppendState*)PyLong_AsVoidPtr(a[0]);
    const long long row = PyLong_AsLongLong(a[3]), pos = PyLong_AsLongLong(a[4]);
    if (PyErr_Occurred() || !st) {
      PyErr_Clear();
      return none();
    }
    const at::Tensor &k = THPVariable_Unpack(a[1]), &v = THPVariable_Unpack(a[2]);
    if (!k.is_cuda() || !v.is_cuda() || k.get_device() != st->device || v.get_device() != st->device) return none();
    if (dtype_code(k.scalar_type()) != st->code || v.scalar_type() != k.scalar_type() || !st->vq) return none();
    kvq_rows kr, vr;
    if (!rows_of(k, &kr) || !rows_of(v, &vr) || k.sizes() != v.sizes()) return none();
    const int64_t L = k.size(2), D = k.size(3);
    if (k.size(0) != st->B || k.size(1) != st->H || row < 0 || row + L > st->rows || L > INT32_MAX) return none();
    if (D * st->bits / 32 != st->code_words || D / st->group != st->groups) return none();
    int rc;
    {
      Unlocked u;
      if (st->rope) {
        kvq_rope_params rp = *st->rope;
        rp.offset = pos;
        rc = ((RopeAppendFn)st->fn)(&kr, st->kq, &vr, st->vq, &rp, row, (int)st->B, (int)st->H, (int)L, (int)D, st->bits,
                                    st->group, st->code, st->stream);
      } else {
        rc = ((AppendFn)st->fn)(&kr, st->kq, &vr, st->vq, row, (int)st->B, (int)st->H, (int)L, (int)D, st->bits, st->group,
                                st->code, st->stream);
      }
    }
    if (rc != KVQ_OK) return failed(rc);
    Py_RETURN_TRUE;
  } catch (...) {
    return none();
  }
}

// views(keys, values, rows) -> the triples' first `rows` rows, as x[..., :rows, :] of each, or None
PyObject* views(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 3) return none();
  try {
    const long long rows = PyLong_AsLongLong(a[2]);
    if (PyErr_Occurred()) {
      PyErr_Clear();
      return none();
    }
    Triple t[2];
    if (!triple_of(a[0], &t[0]) || !triple_of(a[1], &t[1])) return none();
    PyObject* both = PyTuple_New(2);
    for (int i = 0; i < 2; ++i) {
      PyObject* tr = PyTuple_New(3);
      PyTuple_SET_ITEM(both, i, tr);
      const at::Tensor* x[3] = {&t[i].c, &t[i].s, &t[i].b};
      for (int j = 0; j < 3; ++j) {
        if (x[j]->dim() < 2 || rows < 0 || rows > x[j]->size(-2)) {
          Py_DECREF(both);
          return none();
        }
        PyTuple_SET_ITEM(tr, j, THPVariable_Wrap(x[j]->narrow(-2, 0, rows)));
      }
    }
    return both;
  } catch (...) {
    return none();
  }
}

// bind(decode, prefill, decode_workspace_size, prefill_workspace_size, abi, state_bytes, torch): the library's
// entry points; raises where this module was built against another ABI, AppendState or torch.
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 7) {
    PyErr_SetString(PyExc_TypeError, "bind takes 4 addresses, the ABI version, AppendState's size and torch's version");
    return nullptr;
  }
  const long abi = PyLong_AsLong(a[4]), state = PyLong_AsLong(a[5]);
  const char* torch = PyUnicode_AsUTF8(a[6]);
  if (PyErr_Occurred() || !torch) return nullptr;
  const size_t m = strlen(TORCH_VERSION);
  if (abi != KVQ_ABI_VERSION || state != (long)sizeof(AppendState) || strncmp(torch, TORCH_VERSION, m) ||
      (torch[m] >= '0' && torch[m] <= '9')) {
    PyErr_Format(PyExc_ImportError,
                 "_kvqhost.so was built for ABI version %d, an AppendState of %zu bytes and torch %s; here they are %ld, %ld "
                 "and %s: rebuild it",
                 KVQ_ABI_VERSION, sizeof(AppendState), TORCH_VERSION, abi, state, torch);
    return nullptr;
  }
  g.decode = (AttnFn)PyLong_AsVoidPtr(a[0]);
  g.prefill = (AttnFn)PyLong_AsVoidPtr(a[1]);
  g.decode_ws = (SizeFn)PyLong_AsVoidPtr(a[2]);
  g.prefill_ws = (SizeFn)PyLong_AsVoidPtr(a[3]);
  if (PyErr_Occurred()) return nullptr;
  return none();
}

PyMethodDef methods[] = {
    {"attention", (PyCFunction)(void*)attention, METH_FASTCALL, "one quantized attention call"},
    {"append", (PyCFunction)(void*)append, METH_FASTCALL, "one quantize-append"},
    {"views", (PyCFunction)(void*)views, METH_FASTCALL, "the first rows of two triples"},
    {"bind", (PyCFunction)(void*)bind, METH_FASTCALL, "set the library's entry points"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_kvqhost", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__kvqhost() { return PyModule_Create(&module); }
