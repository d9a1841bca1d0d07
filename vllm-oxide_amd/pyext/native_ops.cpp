// Native front end of the Python ops (oxide_paged_kv/_native, a CPython module): checks the tensors,
// allocates outputs and workspaces through torch's allocator and calls the C ABI, for
// the calls of a serving step.  ops.py calls these first; each returns
//   * the op's result,
//   * None when some argument is not of the plain form handled here (a subclass, another
//     dtype or layout, a keyword's other forms): ops.py's general code then runs and
//     raises or handles it,
//   * False when the library recorded an error (ops.py raises it).
//
// Why: a step of a small batch is bound by these calls.  Through ctypes a decode call
// spent 7 of its 13.8 us on attribute reads, argument conversion and torch's stream
// object, around 4.5 us of launches; a layer's three calls 33 us for 16 us of kernels.
//
// The library's entry points are bound by address (bind), so that the functions called
// are those of the library _lib.py loaded.  The GIL is released around library calls.
#include <Python.h>

#include <ATen/Functions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstring>

#include "oxide_paged_kv.h"

namespace {

decltype(&paged_decode_attention) g_decode = nullptr;
decltype(&paged_decode_attention_append) g_decode_append = nullptr;
decltype(&paged_decode_attention_workspace_size) g_decode_ws = nullptr;
decltype(&paged_prefill_attention_workspace) g_prefill_paged = nullptr;
decltype(&varlen_prefill_attention_workspace) g_prefill_varlen = nullptr;
decltype(&prefill_attention_workspace_size) g_prefill_ws = nullptr;
decltype(&qk_norm_rope_and_cache) g_prologue = nullptr;
decltype(&build_decode_metadata_device) g_metadata = nullptr;
decltype(&oxide_last_error) g_last_error = nullptr;

// A plain torch tensor on the device, contiguous.
const at::Tensor* device_tensor(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  return t.defined() && t.is_cuda() && t.layout() == at::kStrided && t.is_contiguous() ? &t : nullptr;
}
bool bits32(const at::Tensor& t) { return t.scalar_type() == at::kInt || t.scalar_type() == at::kUInt32; }
int dtype_code(const at::Tensor& t) {
  return t.scalar_type() == at::kHalf ? OXIDE_DTYPE_F16 : t.scalar_type() == at::kBFloat16 ? OXIDE_DTYPE_BF16 : -1;
}
void* stream_of(const at::Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
bool as_int(PyObject* o, int64_t* v) {
  if (!PyLong_CheckExact(o)) return false;
  int over = 0;
  *v = PyLong_AsLongLongAndOverflow(o, &over);
  return over == 0;
}
bool as_double(PyObject* o, double* v) {
  if (!PyFloat_CheckExact(o)) return false;
  *v = PyFloat_AS_DOUBLE(o);
  return true;
}
// window_left: None = -1, else an int of 32 bits.
bool as_window(PyObject* o, int32_t* v) {
  int64_t x = -1;
  if (o != Py_None && (!as_int(o, &x) || x < INT32_MIN || x > INT32_MAX)) return false;
  *v = static_cast<int32_t>(x);
  return true;
}
// An optional device tensor: false when it is neither None nor one.
bool optional_tensor(PyObject* o, const at::Tensor** t) {
  *t = nullptr;
  return o == Py_None || (*t = device_tensor(o)) != nullptr;
}
void* data(const at::Tensor* t) { return t ? t->data_ptr() : nullptr; }

PyObject* result(at::Tensor t) {
  if (g_last_error() != OXIDE_OK) Py_RETURN_FALSE;
  return THPVariable_Wrap(std::move(t));
}
at::Tensor bytes_like(const at::Tensor& t, int64_t n) { return at::empty({n}, t.options().dtype(at::kByte)); }

// decode(q, k_cache, v_cache, cu_seqlens_k, block_table, max_seqlen_k, softmax_scale,
//        window_left, page_block_size, out, workspace, append)
PyObject* decode(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 12 || !g_decode) Py_RETURN_NONE;
  const at::Tensor *q = device_tensor(a[0]), *k = device_tensor(a[1]), *v = device_tensor(a[2]),
                   *cu = device_tensor(a[3]), *table = device_tensor(a[4]), *out = nullptr, *ws = nullptr;
  int64_t max_k = 0, page = 0;
  double scale = 0;
  int32_t window = -1;
  if (!q || !k || !v || !cu || !table || !as_int(a[5], &max_k) || !as_double(a[6], &scale) ||
      !as_window(a[7], &window) || !as_int(a[8], &page) || !optional_tensor(a[9], &out) ||
      !optional_tensor(a[10], &ws))
    Py_RETURN_NONE;
  const int code = dtype_code(*q);
  if (code < 0 || q->dim() != 3 || k->dim() != 4 || k->sizes() != v->sizes() || k->size(3) != q->size(2) ||
      k->size(1) != page || table->dim() != 2 || table->scalar_type() != at::kInt || !bits32(*cu) ||
      k->scalar_type() != q->scalar_type() || v->scalar_type() != q->scalar_type())
    Py_RETURN_NONE;
  const int64_t B = q->size(0), Hq = q->size(1), D = q->size(2), NB = k->size(0), Hkv = k->size(2);
  const at::Tensor *key = nullptr, *value = nullptr, *slots = nullptr;
  if (a[11] != Py_None) {
    if (!PyTuple_CheckExact(a[11]) || PyTuple_GET_SIZE(a[11]) != 3) Py_RETURN_NONE;
    key = device_tensor(PyTuple_GET_ITEM(a[11], 0));
    value = device_tensor(PyTuple_GET_ITEM(a[11], 1));
    slots = device_tensor(PyTuple_GET_ITEM(a[11], 2));
    if (!key || !value || !slots || key->sizes() != at::IntArrayRef({B, Hkv, D}) || value->sizes() != key->sizes() ||
        slots->scalar_type() != at::kLong)
      Py_RETURN_NONE;
  }
  at::Tensor o = out ? *out : at::empty_like(*q);
  const int64_t need = static_cast<int64_t>(g_decode_ws(B, Hq, Hkv, D, max_k));
  at::Tensor w = ws && static_cast<int64_t>(ws->nbytes()) >= need ? *ws : bytes_like(*q, need > 0 ? need : 1);
  void* s = stream_of(*q);
  void *po = o.data_ptr(), *pq = q->data_ptr(), *pk = k->data_ptr(), *pv = v->data_ptr(), *pw = w.data_ptr();
  const uint32_t* pc = static_cast<const uint32_t*>(cu->data_ptr());
  const int32_t* pt = static_cast<const int32_t*>(table->data_ptr());
  const int64_t width = table->size(1);
  const size_t wbytes = w.nbytes();
  void *pkey = data(key), *pvalue = data(value);
  const int64_t* pslots = static_cast<const int64_t*>(data(slots));
  Py_BEGIN_ALLOW_THREADS;
  if (key)
    g_decode_append(po, pq, pkey, pvalue, pslots, pk, pv, pc, pt, width, NB, B, Hq, Hkv, D, page, max_k, window,
                    static_cast<float>(scale), pw, wbytes, code, s);
  else
    g_decode(po, pq, pk, pv, pc, pt, width, NB, B, Hq, Hkv, D, page, max_k, window, static_cast<float>(scale), pw,
             wbytes, code, s);
  Py_END_ALLOW_THREADS;
  return result(std::move(o));
  END_HANDLE_TH_ERRORS
}

// prefill(q, k, v, cu_seqlens_q, cu_seqlens_k, max_seqlen_q, max_seqlen_k, softmax_scale,
//         block_table, window_left, out)
PyObject* prefill(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 11 || !g_prefill_paged) Py_RETURN_NONE;
  const at::Tensor *q = device_tensor(a[0]), *k = device_tensor(a[1]), *v = device_tensor(a[2]),
                   *cq = device_tensor(a[3]), *ck = device_tensor(a[4]), *table = nullptr, *out = nullptr;
  int64_t max_q = 0, max_k = 0;
  double scale = 0;
  int32_t window = -1;
  if (!q || !k || !v || !cq || !ck || !as_int(a[5], &max_q) || !as_int(a[6], &max_k) || !as_double(a[7], &scale) ||
      !optional_tensor(a[8], &table) || !as_window(a[9], &window) || !optional_tensor(a[10], &out))
    Py_RETURN_NONE;
  const int code = dtype_code(*q);
  const int64_t kd = table ? 4 : 3;
  if (code < 0 || q->dim() != 3 || k->dim() != kd || k->sizes() != v->sizes() || k->size(kd - 1) != q->size(2) ||
      !bits32(*cq) || !bits32(*ck) || cq->dim() != 1 || cq->numel() < 1 || ck->sizes() != cq->sizes() ||
      k->scalar_type() != q->scalar_type() || v->scalar_type() != q->scalar_type() ||
      (table && (table->dim() != 2 || table->scalar_type() != at::kInt)))
    Py_RETURN_NONE;
  const int64_t B = cq->size(0) - 1, Hq = q->size(1), D = q->size(2), Hkv = k->size(kd - 2);
  at::Tensor o = out ? *out : at::empty_like(*q);
  size_t need = g_prefill_ws(B, Hq, Hkv, D, max_q, max_k, window);
  at::Tensor w;
  try {
    if (need > 0) w = bytes_like(*q, static_cast<int64_t>(need));
  } catch (const c10::OutOfMemoryError&) {  // it attends without one
    need = 0;
  }
  void* s = stream_of(*q);
  void *po = o.data_ptr(), *pq = q->data_ptr(), *pk = k->data_ptr(), *pv = v->data_ptr();
  void* pw = need > 0 ? w.data_ptr() : nullptr;
  const uint32_t* pcq = static_cast<const uint32_t*>(cq->data_ptr());
  const uint32_t* pck = static_cast<const uint32_t*>(ck->data_ptr());
  const int32_t* pt = static_cast<const int32_t*>(data(table));
  const int64_t width = table ? table->size(1) : 0, rows = k->size(0), page = table ? k->size(1) : 1;
  Py_BEGIN_ALLOW_THREADS;
  if (table)
    g_prefill_paged(po, pq, pk, pv, pcq, pck, pt, width, rows, B, Hq, Hkv, D, page, max_q, max_k, window,
                    static_cast<float>(scale), pw, need, code, s);
  else
    g_prefill_varlen(po, pq, pk, pv, pcq, pck, rows, B, Hq, Hkv, D, max_q, max_k, window, static_cast<float>(scale),
                     pw, need, code, s);
  Py_END_ALLOW_THREADS;
  return result(std::move(o));
  END_HANDLE_TH_ERRORS
}

// prologue(qkv, num_heads, num_kv_heads, q_norm_weight, k_norm_weight, eps, cos_sin_cache,
//          positions, key_cache, value_cache, slot_mapping, q_out)
PyObject* prologue(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 12 || !g_prologue) Py_RETURN_NONE;
  const at::Tensor *qkv = device_tensor(a[0]), *qw = nullptr, *kw = nullptr, *rope = device_tensor(a[6]),
                   *pos = device_tensor(a[7]), *kc = nullptr, *vc = nullptr, *slots = nullptr, *out = nullptr;
  int64_t Hq = 0, Hkv = 0;
  double eps = 0;
  if (!qkv || !rope || !pos || !as_int(a[1], &Hq) || !as_int(a[2], &Hkv) || !optional_tensor(a[3], &qw) ||
      !optional_tensor(a[4], &kw) || !as_double(a[5], &eps) || !optional_tensor(a[8], &kc) ||
      !optional_tensor(a[9], &vc) || !optional_tensor(a[10], &slots) || !optional_tensor(a[11], &out))
    Py_RETURN_NONE;
  const int code = dtype_code(*qkv);
  if (code < 0 || qkv->dim() != 2 || qkv->stride(1) != 1 || rope->dim() != 2 || rope->scalar_type() != at::kFloat ||
      pos->scalar_type() != at::kInt || (slots && slots->scalar_type() != at::kLong) || Hq < 0 || Hkv < 0)
    Py_RETURN_NONE;
  const int64_t T = qkv->size(0), D = rope->size(1);
  if (out && (out->sizes() != at::IntArrayRef({T, Hq, D}) || out->scalar_type() != qkv->scalar_type() ||
              out->device() != qkv->device()))
    Py_RETURN_NONE;
  at::Tensor o = out ? *out : at::empty({T, Hq, D}, qkv->options());
  void* s = stream_of(*qkv);
  void *po = o.data_ptr(), *px = qkv->data_ptr(), *pqw = data(qw), *pkw = data(kw), *pkc = data(kc), *pvc = data(vc);
  const float* pr = static_cast<const float*>(rope->data_ptr());
  const int32_t* pp = static_cast<const int32_t*>(pos->data_ptr());
  const int64_t* ps = static_cast<const int64_t*>(data(slots));
  const int64_t stride = qkv->stride(0), max_position = rope->size(0);
  Py_BEGIN_ALLOW_THREADS;
  g_prologue(po, nullptr, px, stride, pqw, pkw, eps, pr, max_position, pp, pkc, pvc, ps, T, Hq, Hkv, D, code, s);
  Py_END_ALLOW_THREADS;
  return result(std::move(o));
  END_HANDLE_TH_ERRORS
}

// metadata(context_lens, block_table, block_size) -> (cu_seqlens_k, slot_mapping)
PyObject* metadata(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 3 || !g_metadata) Py_RETURN_NONE;
  const at::Tensor *lens = device_tensor(a[0]), *table = device_tensor(a[1]);
  int64_t page = 0;
  if (!lens || !table || !as_int(a[2], &page) || !bits32(*lens) || lens->dim() != 1 || lens->numel() < 1 ||
      table->dim() != 2 || table->numel() < 1 || table->scalar_type() != at::kInt)
    Py_RETURN_NONE;
  const int64_t B = lens->size(0), width = table->size(1);
  at::Tensor cu = at::empty({B + 1}, lens->options().dtype(at::kInt));
  at::Tensor slots = at::empty({B}, lens->options().dtype(at::kLong));
  void* s = stream_of(*lens);
  const uint32_t* pl = static_cast<const uint32_t*>(lens->data_ptr());
  const int32_t* pt = static_cast<const int32_t*>(table->data_ptr());
  uint32_t* pc = static_cast<uint32_t*>(cu.data_ptr());
  int64_t* ps = static_cast<int64_t*>(slots.data_ptr());
  Py_BEGIN_ALLOW_THREADS;
  g_metadata(pl, pt, width, B, page, pc, ps, s);
  Py_END_ALLOW_THREADS;
  if (g_last_error() != OXIDE_OK) Py_RETURN_FALSE;
  PyObject* c = THPVariable_Wrap(std::move(cu));
  PyObject* m = THPVariable_Wrap(std::move(slots));
  PyObject* both = c && m ? PyTuple_Pack(2, c, m) : nullptr;
  Py_XDECREF(c);
  Py_XDECREF(m);
  return both;
  END_HANDLE_TH_ERRORS
}

// bind(name, address): the library's function of that name; names not used here are
// accepted.
PyObject* bind(PyObject*, PyObject* args) {
  const char* name = nullptr;
  unsigned long long addr = 0;
  if (!PyArg_ParseTuple(args, "sK", &name, &addr)) return nullptr;
  void* p = reinterpret_cast<void*>(static_cast<uintptr_t>(addr));
#define OXIDE_BIND(var, fn) \
  if (std::strcmp(name, #fn) == 0) var = reinterpret_cast<decltype(&fn)>(p);
  OXIDE_BIND(g_decode, paged_decode_attention)
  OXIDE_BIND(g_decode_append, paged_decode_attention_append)
  OXIDE_BIND(g_decode_ws, paged_decode_attention_workspace_size)
  OXIDE_BIND(g_prefill_paged, paged_prefill_attention_workspace)
  OXIDE_BIND(g_prefill_varlen, varlen_prefill_attention_workspace)
  OXIDE_BIND(g_prefill_ws, prefill_attention_workspace_size)
  OXIDE_BIND(g_prologue, qk_norm_rope_and_cache)
  OXIDE_BIND(g_metadata, build_decode_metadata_device)
  OXIDE_BIND(g_last_error, oxide_last_error)
#undef OXIDE_BIND
  Py_RETURN_NONE;
}

template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
PyMethodDef fast(const char* name) {
  return {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(F)), METH_FASTCALL, nullptr};
}
PyMethodDef kMethods[] = {fast<decode>("decode"),     fast<prefill>("prefill"),
                          fast<prologue>("prologue"), fast<metadata>("metadata"),
                          {"bind", bind, METH_VARARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native() {
  PyObject* m = PyModule_Create(&kModule);
  // The torch whose headers it was built against; _lib.py uses it with no other.
  if (m && PyModule_AddStringConstant(m, "torch_version", OXIDE_TORCH_VERSION) < 0) Py_CLEAR(m);
  return m;
}
