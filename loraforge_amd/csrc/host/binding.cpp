// Native call path of the Python operators (loraforge_amd/ops).
//
// Each function takes an operator's arguments, verifies every condition the
// operator's Python checks verify and makes the C-ABI call; on anything out of
// the ordinary (a failed check, a workspace to be grown, another device, a
// tensor subclass or functorch wrapper, ...) it returns None and touches
// nothing, and the operator's own Python code decides what happens: the error
// to raise, or the slower way to serve the call. So it accepts a subset of what
// the operators accept and refuses nothing by itself.
//
// An eager call of the fused linear spent 29 us on the host in about fifty
// small Python checks and ctypes conversions, twice the time of a decode
// kernel at 4096 x 4096; this path takes 6 us.
//
// The library's entry points are handed over as addresses (init), so this
// module binds to whatever build of the library the process loaded.
#include <Python.h>

#include <cstring>

#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ATen.h>

#include "../../../include/loraforge_amd.h"

namespace {

// ---- the library ----------------------------------------------------------
decltype(&lf_nf4_lora_linear) g_linear;
decltype(&lf_nf4_lora_workspace_size) g_linear_ws;
decltype(&lf_lora_apply) g_apply;
decltype(&lf_row_shrink) g_shrink;
decltype(&lf_row_shrink_workspace_size) g_shrink_ws;
decltype(&lf_row_expand) g_expand;
decltype(&lf_nf4_dequant) g_dequant;
decltype(&lf_nf4_dequant_dq_checked) g_dequant_dq;
decltype(&lf_last_error) g_last_error;

PyObject* g_raw_stream;   // torch._C._cuda_getCurrentRawStream
PyObject* g_get_device;   // torch._C._cuda_getDevice
PyObject* g_arch_ok;      // device index -> whether the kernels run there
PyObject* g_workspaces;   // the operators' workspace cache
PyObject* g_multi_cus;    // device index -> compute units
PyObject* g_lora_batch;   // ops.fused.LoraBatch

#define NAMES(X)                                                                                                     \
  X(absmax) X(shape) X(code) X(blocksize) X(quant_type) X(offset) X(state2) X(nested) X(_lf_prepared_scales)         \
  X(a_store) X(a_offsets) X(b_store) X(b_offsets) X(b_strides) X(ranks) X(scales) X(token_slots) X(slice_offsets)    \
  X(max_rank) X(rows)
#define DECL(n) PyObject* s_##n;
NAMES(DECL)
#undef DECL

// An owned reference.
struct Ref {
  PyObject* p;
  explicit Ref(PyObject* o = nullptr) : p(o) {}
  Ref(const Ref&) = delete;
  ~Ref() { Py_XDECREF(p); }
  explicit operator bool() const { return p != nullptr; }
};

PyObject* decline() {
  PyErr_Clear();
  Py_RETURN_NONE;
}

// A HIP error of a library call, with the library's text (as _lib.check raises it).
PyObject* failed() {
  const char* text = g_last_error();
  Ref message(PyUnicode_DecodeUTF8(text, Py_ssize_t(strlen(text)), "replace"));
  if (message) PyErr_SetObject(PyExc_RuntimeError, message.p);
  return nullptr;
}

// The tensor behind a Python object if it is an ordinary dense GPU tensor
// without gradient (an exact torch.Tensor or Parameter: subclasses and
// functorch wrappers have Python or batching semantics of their own).
const at::Tensor* plain(PyObject* o) {
  if (!o || !THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || t.requires_grad()) return nullptr;
  using K = c10::DispatchKey;
  const c10::DispatchKeySet odd{K::Python, K::FuncTorchBatched, K::FuncTorchGradWrapper, K::Functionalize, K::Batched,
                                K::Conjugate, K::Negative, K::ZeroTensor};
  if (t.key_set().has_any(odd) || !t.has_storage()) return nullptr;
  return &t;
}

// Whether a fresh output is memory on the GPU (a dispatch mode may have made something else of it).
bool on_gpu(const at::Tensor& t) {
  return t.is_cuda() && t.has_storage() && !t.key_set().has(c10::DispatchKey::Python) && t.storage().data() != nullptr;
}

bool aligned16(const at::Tensor& t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15u) == 0; }

// A contiguous vector of a type (and, if >= 0, a length) on a device.
const at::Tensor* vec(PyObject* o, at::ScalarType type, const at::Device& dev, int64_t size = -1) {
  const at::Tensor* t = plain(o);
  if (!t || t->dim() != 1 || t->scalar_type() != type || t->device() != dev || !t->is_contiguous()) return nullptr;
  if (t->numel() >= (int64_t(1) << 31) || (size >= 0 && t->numel() != size)) return nullptr;
  return t;
}

const at::Tensor* matrix(PyObject* o, const at::Device& dev) {
  const at::Tensor* t = plain(o);
  if (!t || t->dim() != 2 || t->scalar_type() != at::kBFloat16 || t->device() != dev) return nullptr;
  if (t->size(0) >= (int64_t(1) << 31) || t->size(1) >= (int64_t(1) << 31)) return nullptr;
  return t;
}

bool shares(const at::Tensor& out, std::initializer_list<const at::Tensor*> inputs) {
  const void* p = out.storage().data();
  if (!out.numel()) return false;
  for (const at::Tensor* t : inputs)
    if (t && t->numel() && t->storage().data() == p) return true;
  return false;
}

// Whether the kernels run on `dev` and it is the current device; its current stream.
bool current(const at::Device& dev, void** stream) {
  Ref index(PyLong_FromLong(dev.index()));
  if (!index) return false;
  PyObject* ok = PyDict_GetItem(g_arch_ok, index.p);
  if (ok != Py_True) return false;
  Ref now(PyObject_CallNoArgs(g_get_device));
  if (!now || PyLong_AsLong(now.p) != dev.index()) return false;
  Ref s(PyObject_CallOneArg(g_raw_stream, index.p));
  if (!s) return false;
  *stream = PyLong_AsVoidPtr(s.p);
  return !PyErr_Occurred();
}

// The cached workspace of the current stream, if it holds `need` bytes (else undefined).
// (A reference of its own: the call is made without the GIL.)
at::Tensor workspace(const at::Device& dev, void* stream, int64_t need, PyObject* kind) {
  Ref index(PyLong_FromLong(dev.index()));
  Ref s(PyLong_FromVoidPtr(stream));
  Ref key(kind ? PyTuple_Pack(3, kind, index.p, s.p) : PyTuple_Pack(2, index.p, s.p));
  if (!key) return {};
  PyObject* ws = PyDict_GetItem(g_workspaces, key.p);
  if (!ws || !THPVariable_CheckExact(ws)) return {};
  const at::Tensor& t = THPVariable_Unpack(ws);
  return t.numel() >= need ? t : at::Tensor();
}

bool small_int(PyObject* o, long lo, long hi, long* out) {
  if (!o || !PyLong_CheckExact(o)) return false;
  *out = PyLong_AsLong(o);
  return !PyErr_Occurred() && *out >= lo && *out <= hi;
}

// A library call without the GIL: a launch blocks while the stream's queue is
// full, which must not stop the process's other Python threads (one of them may
// be what the queue waits for). What the call reads is referenced by the caller
// or held above it.
template <class F>
int unlocked(F&& call) {
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = call();
  Py_END_ALLOW_THREADS
  return rc;
}

template <class T>
T* ptr(const at::Tensor* t) {
  return t ? static_cast<T*>(t->data_ptr()) : nullptr;
}

// The C descriptor of a LoraBatch (its fields as ops.fused._lora_struct checks them).
// A subclass or another object may have a num_slices of its own: the Python path's.
struct LoraArg {
  lf_lora d{};
  int slices = 1;
  // The batch's attributes stay referenced until the call is made.
  PyObject* held[10] = {};
  ~LoraArg() {
    for (PyObject* o : held) Py_XDECREF(o);
  }
  bool take(PyObject* b, int64_t m, const at::Device& dev) {
    if (reinterpret_cast<PyObject*>(Py_TYPE(b)) != g_lora_batch) return false;
    PyObject* names[10] = {s_a_store, s_a_offsets, s_b_store, s_b_offsets, s_b_strides,
                           s_ranks,   s_scales,    s_token_slots, s_slice_offsets, s_max_rank};
    for (int i = 0; i < 10; ++i)
      if (!(held[i] = PyObject_GetAttr(b, names[i]))) return false;
    long max_rank;
    if (!small_int(held[9], 1, 64, &max_rank)) return false;
    const at::Tensor* a = vec(held[0], at::kBFloat16, dev);
    const at::Tensor* bs = vec(held[2], at::kBFloat16, dev);
    const at::Tensor* ranks = vec(held[5], at::kInt, dev);
    if (!a || !bs || !ranks || !aligned16(*a) || !aligned16(*bs)) return false;
    const int64_t g = ranks->numel();
    const at::Tensor* ao = vec(held[1], at::kLong, dev, g);
    const at::Tensor* bo = vec(held[3], at::kLong, dev, g);
    const at::Tensor* st = vec(held[4], at::kInt, dev, g);
    const at::Tensor* sc = vec(held[6], at::kFloat, dev, g);
    const at::Tensor* ts = vec(held[7], at::kInt, dev, m);
    const at::Tensor* so = vec(held[8], at::kInt, dev);
    if (!ao || !bo || !st || !sc || !ts || !so || so->numel() < 2 || so->numel() > 4) return false;
    slices = int(so->numel()) - 1;
    d.a_store = ptr<uint16_t>(a);
    d.a_offsets = ptr<int64_t>(ao);
    d.b_store = ptr<uint16_t>(bs);
    d.b_offsets = ptr<int64_t>(bo);
    d.b_strides = ptr<int32_t>(st);
    d.ranks = ptr<int32_t>(ranks);
    d.scales = ptr<float>(sc);
    d.token_slots = ptr<int32_t>(ts);
    d.slice_offsets = ptr<int32_t>(so);
    d.num_slices = slices;
    d.max_rank = int32_t(max_rank);
    d.num_slots = int32_t(g);
    return true;
  }
};

// One entry of a prepared-scales version key against the tensor it stands for.
bool same_version(PyObject* entry, PyObject* tensor) {
  const at::Tensor* t = plain(tensor);
  if (!t || !PyTuple_CheckExact(entry) || PyTuple_GET_SIZE(entry) != 2 || t->is_inference()) return false;
  PyObject* version = PyTuple_GET_ITEM(entry, 1);
  if (!PyLong_CheckExact(version)) return false;
  return PyLong_AsVoidPtr(PyTuple_GET_ITEM(entry, 0)) == t->data_ptr() &&
         PyLong_AsLongLong(version) == int64_t(t->_version()) && !PyErr_Occurred();
}

// The fp32 block scales of a call with scales=None: the state's own, or the
// prepared ones of a nested state while its version key holds (ops.fused.scale_key).
PyObject* state_scales(PyObject* qweight, PyObject* state, PyObject* absmax, PyObject* code) {
  Ref nested(PyObject_GetAttr(state, s_nested));
  if (!nested) return nullptr;
  if (nested.p == Py_False) {
    Py_INCREF(absmax);
    return absmax;
  }
  if (nested.p != Py_True) return nullptr;
  Ref cached(PyObject_GetAttr(state, s__lf_prepared_scales));
  if (!cached || !PyTuple_CheckExact(cached.p) || PyTuple_GET_SIZE(cached.p) != 2) return nullptr;
  PyObject* key = PyTuple_GET_ITEM(cached.p, 0);
  if (!PyTuple_CheckExact(key) || PyTuple_GET_SIZE(key) != 2) return nullptr;
  if (PyLong_AsVoidPtr(PyTuple_GET_ITEM(key, 0)) != state) return nullptr;
  PyObject* parts = PyTuple_GET_ITEM(key, 1);
  if (!PyTuple_CheckExact(parts) || PyTuple_GET_SIZE(parts) != 6) return nullptr;
  Ref two(PyObject_GetAttr(state, s_state2));
  Ref offset(PyObject_GetAttr(state, s_offset));
  if (!two || !offset) return nullptr;
  Ref absmax2(PyObject_GetAttr(two.p, s_absmax));
  Ref code2(PyObject_GetAttr(two.p, s_code));
  if (!absmax2 || !code2) return nullptr;
  PyObject* now[6] = {qweight, absmax, code, absmax2.p, code2.p, offset.p};
  for (int i = 0; i < 6; ++i)
    if (!same_version(PyTuple_GET_ITEM(parts, i), now[i])) return nullptr;
  PyObject* scales = PyTuple_GET_ITEM(cached.p, 1);
  Py_INCREF(scales);
  return scales;
}

// The double-quant part of a weight descriptor (ops.fused._weight_struct's checks).
struct NestedArg {
  PyObject* held[5] = {};
  ~NestedArg() {
    for (PyObject* o : held) Py_XDECREF(o);
  }
  bool take(PyObject* state, PyObject* absmax_o, int64_t blocks, const at::Device& dev, lf_nf4_weight* w) {
    PyObject* two = held[0] = PyObject_GetAttr(state, s_state2);
    if (!two || !(held[1] = PyObject_GetAttr(state, s_offset)) || !(held[2] = PyObject_GetAttr(two, s_absmax)) ||
        !(held[3] = PyObject_GetAttr(two, s_code)) || !(held[4] = PyObject_GetAttr(two, s_blocksize)))
      return false;
    long block;
    if (!small_int(held[4], 1, 1 << 30, &block)) return false;
    const at::Tensor* absmax = plain(absmax_o);
    const at::Tensor* offset = plain(held[1]);
    const at::Tensor* absmax2 = plain(held[2]);
    const at::Tensor* code2 = plain(held[3]);
    if (!absmax || !offset || !absmax2 || !code2 || absmax->device() != dev || offset->device() != dev ||
        absmax2->device() != dev || code2->device() != dev)
      return false;
    if (absmax->scalar_type() != at::kByte || absmax->numel() != blocks || !absmax->is_contiguous() ||
        absmax2->scalar_type() != at::kFloat || !absmax2->is_contiguous() ||
        absmax2->numel() != (blocks + block - 1) / block || code2->scalar_type() != at::kFloat || code2->numel() != 256 ||
        !code2->is_contiguous() || offset->scalar_type() != at::kFloat || offset->numel() != 1)
      return false;
    w->absmax_q = ptr<uint8_t>(absmax);
    w->absmax2 = ptr<float>(absmax2);
    w->code2 = ptr<float>(code2);
    w->offset = ptr<float>(offset);
    w->dq_block = block;
    return true;
  }
};

// linear(x, qweight, state, scales, bias, lora, out, exact, swiglu, flags) -> out or None
PyObject* linear(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 10) return decline();
  PyObject *py_x = args[0], *py_q = args[1], *state = args[2], *py_scales = args[3], *py_bias = args[4];
  PyObject *py_lora = args[5], *py_out = args[6];
  const bool exact = args[7] == Py_True, swiglu = args[8] == Py_True;
  if ((!exact && args[7] != Py_False) || (!swiglu && args[8] != Py_False)) return decline();
  long flags;
  if (!small_int(args[9], 0, 1 << 16, &flags)) return decline();
  const at::Tensor* x = plain(py_x);
  const at::Tensor* q = plain(py_q);
  if (!x || !q) return decline();
  const at::Device dev = x->device();

  Ref quant_type(PyObject_GetAttr(state, s_quant_type)), blocksize(PyObject_GetAttr(state, s_blocksize));
  Ref shape(PyObject_GetAttr(state, s_shape)), absmax(PyObject_GetAttr(state, s_absmax));
  Ref code_o(PyObject_GetAttr(state, s_code));
  if (!quant_type || !blocksize || !shape || !absmax || !code_o) return decline();
  if (!PyUnicode_Check(quant_type.p) || PyUnicode_CompareWithASCIIString(quant_type.p, "nf4") != 0) return decline();
  long bs, n, k;
  if (!small_int(blocksize.p, 64, 64, &bs)) return decline();
  if (!PyTuple_Check(shape.p) || PyTuple_GET_SIZE(shape.p) != 2) return decline();
  if (!small_int(PyTuple_GET_ITEM(shape.p, 0), 64, 1 << 28, &n) || !small_int(PyTuple_GET_ITEM(shape.p, 1), 64, 1 << 28, &k))
    return decline();
  if (n % 64 || k % 64) return decline();
  if (x->scalar_type() != at::kBFloat16 || x->dim() < 1 || x->size(-1) != k || x->stride(-1) != 1) return decline();
  const bool flat = x->dim() == 2;
  if (!flat && !x->is_contiguous()) return decline();
  const int64_t m = x->numel() / k;
  const int64_t x_stride = flat ? x->stride(0) : k;
  if (m == 0 || x_stride < k || x_stride % 8 || !aligned16(*x)) return decline();
  if (q->device() != dev || q->scalar_type() != at::kByte || q->numel() != int64_t(n) * k / 2 || !q->is_contiguous() ||
      !aligned16(*q))
    return decline();
  const at::Tensor* bias = nullptr;
  if (py_bias != Py_None && !(bias = vec(py_bias, at::kBFloat16, dev, n))) return decline();
  const at::Tensor* code = plain(code_o.p);
  if (!code || code->device() != dev || code->scalar_type() != at::kFloat || code->numel() != 16 || !code->is_contiguous())
    return decline();

  // Block scales: the caller's, the state's (prepared ones for a nested state)
  // or, on request and for exact prefill calls, the nested state itself.
  lf_nf4_weight w{};
  Ref nested(PyObject_GetAttr(state, s_nested));
  if (!nested || (nested.p != Py_True && nested.p != Py_False)) return decline();
  bool from_state = false;
  if (PyUnicode_Check(py_scales)) {
    if (nested.p != Py_True || PyUnicode_CompareWithASCIIString(py_scales, "nested") != 0) return decline();
    from_state = true;
  } else if (py_scales == Py_None) {
    from_state = nested.p == Py_True && m > 64 && exact && !(flags & LF_PLAN_DECODE_CHUNKS);
  }
  Ref scales_o(from_state                ? nullptr
               : py_scales != Py_None ? (Py_INCREF(py_scales), py_scales)
                                         : state_scales(py_q, state, absmax.p, code_o.p));
  NestedArg two;
  if (from_state) {
    if (!two.take(state, absmax.p, int64_t(n) * k / 64, dev, &w)) return decline();
  } else {
    const at::Tensor* scales = plain(scales_o.p);
    if (!scales || scales->device() != dev || scales->scalar_type() != at::kFloat || !scales->is_contiguous() ||
        scales->numel() != int64_t(n) * k / 64)
      return decline();
    w.scales = ptr<float>(scales);
  }

  LoraArg lora;
  const bool has_lora = py_lora != Py_None;
  if (has_lora && !lora.take(py_lora, m, dev)) return decline();
  if (swiglu && has_lora && lora.slices != 2) return decline();
  const int64_t width = swiglu ? n / 2 : n;

  void* stream;
  if (!current(dev, &stream)) return decline();
  const int64_t need = g_linear_ws(m, n, k, has_lora ? lora.slices : 1, has_lora ? lora.d.max_rank : 1);
  if (need < 0) return decline();
  const at::Tensor ws = workspace(dev, stream, need, nullptr);
  if (!ws.defined()) return decline();

  at::Tensor result;
  int64_t y_stride = width;
  if (py_out != Py_None) {
    const at::Tensor* out = plain(py_out);
    // (The SwiGLU output above 64 tokens has alignment rules of its own.)
    if (!out || !flat || out->dim() != 2 || out->scalar_type() != at::kBFloat16 || out->device() != dev ||
        out->size(0) != m || out->size(1) != width || out->stride(1) != 1 || (swiglu && m > 64) ||
        shares(*out, {x, q, bias}))
      return decline();
    if (m > 1 && out->stride(0) < width) return decline();
    result = *out;
    y_stride = out->stride(0);
    if (y_stride < width) return decline();
  } else {
    std::vector<int64_t> sizes(x->sizes().begin(), x->sizes().end());
    sizes.back() = width;
    result = at::empty(sizes, x->options());
    if (!on_gpu(result)) return decline();
  }
  w.qweight = ptr<uint8_t>(q);
  w.code = ptr<float>(code);
  w.n = n;
  w.k = k;
  const int rc = unlocked([&] {
    return g_linear(ptr<uint16_t>(x), m, x_stride, &w, ptr<uint16_t>(bias), has_lora ? &lora.d : nullptr,
                    static_cast<uint16_t*>(result.data_ptr()), y_stride, ws.data_ptr(), ws.numel(),
                    int32_t(flags) | (exact ? LF_EXACT_WEIGHTS : 0) | (swiglu ? LF_SWIGLU_OUTPUT : 0), stream);
  });
  if (rc == LF_EINVAL) return decline();  // (nothing was launched; the Python path raises the message)
  if (rc != LF_OK) return failed();
  if (py_out != Py_None) {
    Py_INCREF(py_out);
    return py_out;
  }
  return THPVariable_Wrap(result);
}

// apply(x, y, lora) -> y or None
PyObject* apply(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 3) return decline();
  const at::Tensor* x = plain(args[0]);
  if (!x) return decline();
  const at::Device dev = x->device();
  x = matrix(args[0], dev);
  const at::Tensor* y = matrix(args[1], dev);
  if (!x || !y) return decline();
  const int64_t m = x->size(0), k = x->size(1), n = y->size(1);
  if (m == 0 || y->size(0) != m || n <= 0 || k <= 0 || n % 64 || k % 64 || x->stride(1) != 1 || y->stride(1) != 1 ||
      x->stride(0) % 8 || !aligned16(*x) || shares(*y, {x}))
    return decline();
  LoraArg lora;
  if (!lora.take(args[2], m, dev)) return decline();
  void* stream;
  if (!current(dev, &stream)) return decline();
  const int64_t need = g_linear_ws(m < 64 ? m : 64, n, k, lora.slices, lora.d.max_rank);
  if (need < 0) return decline();
  const at::Tensor ws = workspace(dev, stream, need, nullptr);
  if (!ws.defined()) return decline();
  const int rc = unlocked([&] {
    return g_apply(ptr<uint16_t>(x), m, x->stride(0), n, k, &lora.d, ptr<uint16_t>(y), y->stride(0), ws.data_ptr(),
                   ws.numel(), 0, stream);
  });
  if (rc == LF_EINVAL) return decline();
  if (rc != LF_OK) return failed();
  Py_INCREF(args[1]);
  return args[1];
}

// shrink(x, a, output, slots, ranks, num_slices, max_rank) -> True or None
PyObject* shrink(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 7) return decline();
  const at::Tensor* x = plain(args[0]);
  if (!x) return decline();
  const at::Device dev = x->device();
  x = matrix(args[0], dev);
  const at::Tensor* a = plain(args[1]);
  const at::Tensor* z = matrix(args[2], dev);
  long slices, max_rank;
  if (!x || !a || !z || !small_int(args[5], 1, 3, &slices) || !small_int(args[6], 1, 64, &max_rank)) return decline();
  if (a->dim() != 3 || a->scalar_type() != at::kBFloat16 || a->device() != dev) return decline();
  const int64_t m = x->size(0), width = x->size(1), g = a->size(0), rows = a->size(1);
  if (m == 0 || g < 1 || g >= (int64_t(1) << 31) || rows >= (int64_t(1) << 31) || rows % slices ||
      rows / slices < max_rank || a->size(2) != width || z->size(0) != m || z->size(1) != rows)
    return decline();
  if (width < 1 || width % 8 || x->stride(1) != 1 || x->stride(0) < width || x->stride(0) % 8 || !aligned16(*x) ||
      !aligned16(*a) || !a->is_contiguous() || !z->is_contiguous())
    return decline();
  const at::Tensor* slots = vec(args[3], at::kInt, dev, m);
  const at::Tensor* ranks = vec(args[4], at::kInt, dev, g);
  if (!slots || !ranks || shares(*z, {x, a, slots, ranks})) return decline();
  void* stream;
  if (!current(dev, &stream)) return decline();
  const int64_t need = g_shrink_ws(m, width, g, int32_t(slices), int32_t(max_rank));
  if (need < 0) return decline();
  const at::Tensor ws = need ? workspace(dev, stream, need, s_rows) : at::Tensor();
  if (need && !ws.defined()) return decline();
  const int rc = unlocked([&] {
    return g_shrink(ptr<uint16_t>(x), ptr<uint16_t>(a), ptr<uint16_t>(z), ptr<int32_t>(slots), ptr<int32_t>(ranks), m,
                    width, x->stride(0), g, int32_t(slices), rows / slices, int32_t(max_rank),
                    need ? ws.data_ptr() : nullptr, need ? ws.numel() : 0, 0, stream);
  });
  if (rc == LF_EINVAL) return decline();
  if (rc != LF_OK) return failed();
  Py_RETURN_TRUE;
}

// expand(z, b, output, b_offsets, b_strides, ranks, scales, segment_indptr, segment_slots, token_indices,
//        slice_offsets, segment_count, blocks, threads) -> True or None
PyObject* expand(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 14) return decline();
  const at::Tensor* z = plain(args[0]);
  if (!z) return decline();
  const at::Device dev = z->device();
  z = matrix(args[0], dev);
  const at::Tensor* b = vec(args[1], at::kBFloat16, dev);
  const at::Tensor* y = matrix(args[2], dev);
  const at::Tensor* ranks = vec(args[5], at::kInt, dev);
  if (!z || !b || !y || !ranks) return decline();
  const int64_t g = ranks->numel();
  const at::Tensor* offsets = vec(args[3], at::kLong, dev, g);
  const at::Tensor* strides = vec(args[4], at::kInt, dev, g);
  const at::Tensor* scales = vec(args[6], at::kFloat, dev, g);
  const at::Tensor* slots = vec(args[8], at::kInt, dev);
  if (!offsets || !strides || !scales || !slots) return decline();
  const at::Tensor* indptr = vec(args[7], at::kInt, dev, slots->numel() + 1);
  const at::Tensor* tokens = vec(args[9], at::kInt, dev);
  const at::Tensor* bounds = vec(args[10], at::kInt, dev);
  const at::Tensor* count = vec(args[11], at::kInt, dev, 1);
  if (!indptr || !tokens || !bounds || !count) return decline();
  const int64_t slices = bounds->numel() - 1, m = z->size(0), n = y->size(1);
  if (m == 0 || g < 1 || slices < 1 || slices > 3 || z->size(1) < slices || z->size(1) % slices || y->size(0) != m || n < 1 ||
      !z->is_contiguous() || !aligned16(*b) || y->stride(1) != 1 || y->stride(0) < n)
    return decline();
  long threads, blocks;
  if (!small_int(args[13], 128, 256, &threads) || (threads != 128 && threads != 256)) return decline();
  if (args[12] == Py_None) {
    Ref index(PyLong_FromLong(dev.index()));
    PyObject* cus = index ? PyDict_GetItem(g_multi_cus, index.p) : nullptr;
    if (!small_int(cus, 1, 32767, &blocks)) return decline();
    blocks *= 2;
  } else if (!small_int(args[12], 1, 65535, &blocks)) {
    return decline();
  }
  if (slots->numel() * ((n + threads - 1) / threads) >= (int64_t(1) << 31)) return decline();
  if (shares(*y, {z, b, offsets, strides, ranks, scales, indptr, slots, tokens, bounds, count})) return decline();
  void* stream;
  if (!current(dev, &stream)) return decline();
  const int rc = unlocked([&] {
    return g_expand(ptr<uint16_t>(z), ptr<uint16_t>(b), ptr<int64_t>(offsets), ptr<int32_t>(strides), ptr<uint16_t>(y),
                    ptr<int32_t>(indptr), ptr<int32_t>(slots), ptr<int32_t>(tokens), ptr<int32_t>(ranks),
                    ptr<float>(scales), ptr<int32_t>(bounds), ptr<int32_t>(count), slots->numel(), m, n, y->stride(0),
                    int32_t(slices), z->size(1) / slices, int32_t(blocks), int32_t(threads), stream);
  });
  if (rc == LF_EINVAL) return decline();
  if (rc != LF_OK) return failed();
  Py_RETURN_TRUE;
}

// dequant(qweight, scales, code, shape) -> out or None
PyObject* dequant(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 4) return decline();
  long n, k;
  if (!PyTuple_CheckExact(args[3]) || PyTuple_GET_SIZE(args[3]) != 2 ||
      !small_int(PyTuple_GET_ITEM(args[3], 0), 64, 1 << 28, &n) || !small_int(PyTuple_GET_ITEM(args[3], 1), 64, 1 << 28, &k) ||
      n % 64 || k % 64)
    return decline();
  const int64_t size = int64_t(n) * k;
  const at::Tensor* q = plain(args[0]);
  const at::Tensor* s = plain(args[1]);
  const at::Tensor* c = plain(args[2]);
  if (!q || !s || !c) return decline();
  const at::Device dev = q->device();
  if (s->device() != dev || c->device() != dev || q->scalar_type() != at::kByte || q->numel() != size / 2 ||
      s->scalar_type() != at::kFloat || s->numel() != size / 64 || c->scalar_type() != at::kFloat || c->numel() != 16 ||
      !q->is_contiguous() || !s->is_contiguous() || !c->is_contiguous())
    return decline();
  void* stream;
  if (!current(dev, &stream)) return decline();
  at::Tensor out = at::empty({n, k}, s->options().dtype(at::kBFloat16));
  if (!on_gpu(out)) return decline();
  const int rc = unlocked([&] {
    return g_dequant(ptr<uint8_t>(q), ptr<float>(s), ptr<float>(c), static_cast<uint16_t*>(out.data_ptr()), size, stream);
  });
  if (rc == LF_EINVAL) return decline();
  if (rc != LF_OK) return failed();
  return THPVariable_Wrap(out);
}

// dequant_nested(qweight, state) -> out or None. The library checks the codebook
// in the kernel: two blocking copies and a comparison launch per call before
// (115 us at 24576 x 4096, the kernel itself 40).
PyObject* dequant_nested(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 2) return decline();
  PyObject* state = args[1];
  const at::Tensor* q = plain(args[0]);
  if (!q) return decline();
  const at::Device dev = q->device();
  Ref nested(PyObject_GetAttr(state, s_nested)), shape(PyObject_GetAttr(state, s_shape));
  Ref absmax(PyObject_GetAttr(state, s_absmax)), code_o(PyObject_GetAttr(state, s_code));
  if (!nested || !shape || !absmax || !code_o || nested.p != Py_True) return decline();
  long n, k;
  if (!PyTuple_Check(shape.p) || PyTuple_GET_SIZE(shape.p) != 2 ||
      !small_int(PyTuple_GET_ITEM(shape.p, 0), 64, 1 << 28, &n) || !small_int(PyTuple_GET_ITEM(shape.p, 1), 64, 1 << 28, &k) ||
      n % 64 || k % 64)
    return decline();
  const int64_t size = int64_t(n) * k;
  const at::Tensor* code = plain(code_o.p);
  if (q->scalar_type() != at::kByte || q->numel() != size / 2 || !q->is_contiguous() || !code || code->device() != dev ||
      code->scalar_type() != at::kFloat || code->numel() != 16 || !code->is_contiguous())
    return decline();
  lf_nf4_weight w{};
  NestedArg two;
  if (!two.take(state, absmax.p, size / 64, dev, &w)) return decline();
  void* stream;
  if (!current(dev, &stream)) return decline();
  at::Tensor out = at::empty({n, k}, code->options().dtype(at::kBFloat16));
  if (!on_gpu(out)) return decline();
  int32_t canonical = 0;
  uint16_t* dst = static_cast<uint16_t*>(out.data_ptr());
  const int rc = unlocked([&] {
    return g_dequant_dq(ptr<uint8_t>(q), w.absmax_q, w.absmax2, w.code2, w.offset, w.dq_block, ptr<float>(code), dst, size,
                        &canonical, stream);
  });
  if (rc == LF_EINVAL || (rc == LF_OK && !canonical)) return decline();
  if (rc != LF_OK) return failed();
  return THPVariable_Wrap(out);
}

// init(addresses, raw_stream, get_device, arch_ok, workspaces, compute_units, lora_batch)
PyObject* init(PyObject*, PyObject* args) {
  PyObject *addresses, *raw, *dev, *arch, *ws, *cus, *batch;
  if (!PyArg_ParseTuple(args, "O!OOO!O!O!O!", &PyTuple_Type, &addresses, &raw, &dev, &PyDict_Type, &arch, &PyDict_Type, &ws,
                        &PyDict_Type, &cus, &PyType_Type, &batch))
    return nullptr;
  constexpr int kEntries = 9;
  void* a[kEntries];
  if (PyTuple_GET_SIZE(addresses) != kEntries) {
    PyErr_SetString(PyExc_ValueError, "nine entry points expected");
    return nullptr;
  }
  for (int i = 0; i < kEntries; ++i)
    if (!(a[i] = PyLong_AsVoidPtr(PyTuple_GET_ITEM(addresses, i)))) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "null entry point");
      return nullptr;
    }
  g_linear = reinterpret_cast<decltype(g_linear)>(a[0]);
  g_linear_ws = reinterpret_cast<decltype(g_linear_ws)>(a[1]);
  g_apply = reinterpret_cast<decltype(g_apply)>(a[2]);
  g_shrink = reinterpret_cast<decltype(g_shrink)>(a[3]);
  g_shrink_ws = reinterpret_cast<decltype(g_shrink_ws)>(a[4]);
  g_expand = reinterpret_cast<decltype(g_expand)>(a[5]);
  g_dequant = reinterpret_cast<decltype(g_dequant)>(a[6]);
  g_dequant_dq = reinterpret_cast<decltype(g_dequant_dq)>(a[7]);
  g_last_error = reinterpret_cast<decltype(g_last_error)>(a[8]);
#define INTERN(n) \
  if (!s_##n && !(s_##n = PyUnicode_InternFromString(#n))) return nullptr;
  NAMES(INTERN)
#undef INTERN
  PyObject** slot[6] = {&g_raw_stream, &g_get_device, &g_arch_ok, &g_workspaces, &g_multi_cus, &g_lora_batch};
  PyObject* value[6] = {raw, dev, arch, ws, cus, batch};
  for (int i = 0; i < 6; ++i) {
    Py_INCREF(value[i]);
    Py_XDECREF(*slot[i]);
    *slot[i] = value[i];
  }
  Py_RETURN_NONE;
}

// A C++ exception (an allocation that fails, say) becomes a Python one.
template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
PyObject* guarded(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  return F(self, args, nargs);
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"init", init, METH_VARARGS, nullptr},
    {"linear", reinterpret_cast<PyCFunction>(guarded<linear>), METH_FASTCALL, nullptr},
    {"apply", reinterpret_cast<PyCFunction>(guarded<apply>), METH_FASTCALL, nullptr},
    {"shrink", reinterpret_cast<PyCFunction>(guarded<shrink>), METH_FASTCALL, nullptr},
    {"expand", reinterpret_cast<PyCFunction>(guarded<expand>), METH_FASTCALL, nullptr},
    {"dequant_nested", reinterpret_cast<PyCFunction>(guarded<dequant_nested>), METH_FASTCALL, nullptr},
    {"dequant", reinterpret_cast<PyCFunction>(guarded<dequant>), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_binding", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__binding() { return PyModule_Create(&module); }
