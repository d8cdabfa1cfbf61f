// Python's side of the C ABI in native code: the device tensor `MiBackend` hands out and a typed call
// for every entry point its methods make.
//
// What bounds a decode step or an op-by-op training step of a small model is this path, not the
// device: some 170 calls per decoded token. Through ctypes a call boxed each argument in an object of
// its own, allocated and freed its output through two more calls and took 12-15 us of host time for
// a 2-5 us kernel. Here an argument is converted straight into the parameter's type (deduced from the
// declaration in ojas_mi355x.h, so there is no second table of signatures), and a tensor's
// allocation, release and views are C.
//
// The library is opened at run time (`load`), so importing this module needs neither it nor a device.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <dlfcn.h>
#include <structmember.h>

#include <cstring>
#include <tuple>
#include <type_traits>
#include <utility>

#include "ojas_mi355x.h"

namespace {

PyObject* g_error = nullptr;  // OjasError(code, detail)
constexpr int kSizes[4] = {4, 2, 4, 1};  // F32, BF16, U32, I8

// ---- the context: an omx_ctx whose handle becomes null when the backend closes ----
struct Context {
  PyObject_HEAD
  omx_ctx* ctx;
};

int32_t (*p_alloc)(omx_ctx*, uint64_t, void**) = nullptr;
int32_t (*p_free)(omx_ctx*, void*) = nullptr;
size_t (*p_last_error)(omx_ctx*, char*, size_t) = nullptr;

PyObject* raise(omx_ctx* ctx, int32_t rc) {
  char buf[512];
  buf[0] = 0;
  if (ctx && p_last_error) p_last_error(ctx, buf, sizeof buf);
  PyObject* text = PyUnicode_DecodeUTF8(buf, static_cast<Py_ssize_t>(strlen(buf)), "replace");
  if (!text) return nullptr;
  PyObject* e = PyObject_CallFunction(g_error ? g_error : PyExc_RuntimeError, "iN", static_cast<int>(rc), text);
  if (!e) return nullptr;
  PyErr_SetObject(reinterpret_cast<PyObject*>(Py_TYPE(e)), e);
  Py_DECREF(e);
  return nullptr;
}

PyObject* raise_text(int32_t rc, const char* text) {
  PyObject* e = PyObject_CallFunction(g_error ? g_error : PyExc_RuntimeError, "is", static_cast<int>(rc), text);
  if (!e) return nullptr;
  PyErr_SetObject(reinterpret_cast<PyObject*>(Py_TYPE(e)), e);
  Py_DECREF(e);
  return nullptr;
}

PyObject* context_new(PyTypeObject* type, PyObject* args, PyObject*) {
  unsigned long long address = 0;
  if (!PyArg_ParseTuple(args, "K", &address)) return nullptr;
  Context* self = reinterpret_cast<Context*>(type->tp_alloc(type, 0));
  if (self) self->ctx = reinterpret_cast<omx_ctx*>(address);
  return reinterpret_cast<PyObject*>(self);
}
PyObject* context_close(PyObject* self, PyObject*) {
  reinterpret_cast<Context*>(self)->ctx = nullptr;
  Py_RETURN_NONE;
}
PyMethodDef context_methods[] = {{"close", context_close, METH_NOARGS, "Forget the handle; tensors no longer free themselves."},
                                 {nullptr, nullptr, 0, nullptr}};
PyTypeObject ContextType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// ---- the device tensor ----
struct Tensor {
  PyObject_HEAD
  Context* context;   // whose device memory this is
  PyObject* backend;  // the MiBackend (None once dropped)
  PyObject* shape;    // tuple of int
  PyObject* base;     // the tensor a view keeps alive
  PyObject* dict;     // attributes a caller gives it (null until one does)
  PyObject* weak;     // weak references to it
  unsigned long long ptr;
  Py_ssize_t numel;
  int dtype;
  char owns, compute_bf16;
};
PyTypeObject TensorType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// Elements of a shape tuple (1 for rank 0); -1 with an error set when an axis is no whole number.
Py_ssize_t elements(PyObject* shape) {
  Py_ssize_t n = 1;
  const Py_ssize_t rank = PyTuple_GET_SIZE(shape);
  for (Py_ssize_t i = 0; i < rank; ++i) {
    const Py_ssize_t axis = PyLong_AsSsize_t(PyTuple_GET_ITEM(shape, i));
    if (axis == -1 && PyErr_Occurred()) return -1;
    n *= axis;
  }
  return n;
}

// A tuple of plain ints from a shape given as a tuple, a list or one number.
PyObject* shape_tuple(PyObject* given) {
  if (PyTuple_CheckExact(given)) {
    const Py_ssize_t rank = PyTuple_GET_SIZE(given);
    bool plain = true;
    for (Py_ssize_t i = 0; i < rank; ++i) plain &= PyLong_CheckExact(PyTuple_GET_ITEM(given, i)) != 0;
    if (plain) {
      Py_INCREF(given);
      return given;
    }
  }
  PyObject* seq = PyIndex_Check(given) ? PyTuple_Pack(1, given) : PySequence_Tuple(given);
  if (!seq) return nullptr;
  PyObject* out = PyTuple_New(PyTuple_GET_SIZE(seq));
  for (Py_ssize_t i = 0; out && i < PyTuple_GET_SIZE(seq); ++i) {
    PyObject* axis = PyNumber_Long(PyTuple_GET_ITEM(seq, i));
    if (!axis) Py_CLEAR(out);
    else PyTuple_SET_ITEM(out, i, axis);
  }
  Py_DECREF(seq);
  return out;
}

Tensor* make_tensor(PyObject* backend, Context* context, unsigned long long ptr, PyObject* shape /* stolen */, Py_ssize_t n,
                    int dtype, bool owns) {
  Tensor* t = reinterpret_cast<Tensor*>(TensorType.tp_alloc(&TensorType, 0));
  if (!t) {
    Py_DECREF(shape);
    return nullptr;
  }
  Py_XINCREF(context);
  Py_INCREF(backend);
  t->context = context;
  t->backend = backend;
  t->shape = shape;
  t->ptr = ptr;
  t->numel = n;
  t->dtype = dtype;
  t->owns = owns;
  return t;
}

// The context of a backend, or null (a new reference).
Context* context_in(PyObject* backend) {
  PyObject* context = backend == Py_None ? nullptr : PyObject_GetAttrString(backend, "_context");
  if (!context) PyErr_Clear();
  if (context && Py_TYPE(context) != &ContextType) Py_CLEAR(context);
  return reinterpret_cast<Context*>(context);
}
// A tensor of no elements and no memory until its __init__ (a subclass may have one of its own).
PyObject* tensor_new(PyTypeObject* type, PyObject*, PyObject*) {
  PyObject* shape = PyTuple_New(0);
  if (!shape) return nullptr;
  Tensor* t = reinterpret_cast<Tensor*>(type->tp_alloc(type, 0));
  if (!t) {
    Py_DECREF(shape);
    return nullptr;
  }
  Py_INCREF(Py_None);
  t->backend = Py_None;
  t->shape = shape;
  t->numel = 1;
  return reinterpret_cast<PyObject*>(t);
}
// DeviceTensor(backend, ptr, shape, dtype, owns=True)
int tensor_init(PyObject* self, PyObject* args, PyObject* kwargs) {
  static const char* names[] = {"backend", "ptr", "shape", "dtype", "owns", nullptr};
  PyObject *backend, *ptr_obj, *given;
  int dtype, owns = 1;
  if (!PyArg_ParseTupleAndKeywords(args, kwargs, "OOOi|p", const_cast<char**>(names), &backend, &ptr_obj, &given, &dtype, &owns))
    return -1;
  unsigned long long ptr = 0;
  if (ptr_obj != Py_None) {
    ptr = PyLong_AsUnsignedLongLong(ptr_obj);
    if (PyErr_Occurred()) return -1;
  }
  PyObject* shape = shape_tuple(given);
  if (!shape) return -1;
  const Py_ssize_t n = elements(shape);
  if (n == -1 && PyErr_Occurred()) {
    Py_DECREF(shape);
    return -1;
  }
  Tensor* t = reinterpret_cast<Tensor*>(self);
  PyObject *old_backend = t->backend, *old_shape = t->shape, *old_context = reinterpret_cast<PyObject*>(t->context);
  Py_INCREF(backend);
  t->backend = backend;
  t->context = context_in(backend);
  t->shape = shape;
  t->ptr = ptr;
  t->numel = n;
  t->dtype = dtype;
  t->owns = owns;
  Py_XDECREF(old_backend);
  Py_XDECREF(old_shape);
  Py_XDECREF(old_context);
  return 0;
}

void tensor_dealloc(PyObject* self) {
  Tensor* t = reinterpret_cast<Tensor*>(self);
  PyObject_GC_UnTrack(self);
  if (t->weak) PyObject_ClearWeakRefs(self);
  if (t->owns && t->ptr && t->context && t->context->ctx && p_free) {
    // A block too large for the context's pool goes back to the driver, which waits for the stream.
    PyThreadState* unlocked = t->numel >= (64l << 20) ? PyEval_SaveThread() : nullptr;
    p_free(t->context->ctx, reinterpret_cast<void*>(t->ptr));
    if (unlocked) PyEval_RestoreThread(unlocked);
  }
  Py_XDECREF(t->context);
  Py_XDECREF(t->backend);
  Py_XDECREF(t->shape);
  Py_XDECREF(t->base);
  Py_XDECREF(t->dict);
  Py_TYPE(self)->tp_free(self);
}
int tensor_traverse(PyObject* self, visitproc visit, void* arg) {
  Tensor* t = reinterpret_cast<Tensor*>(self);
  Py_VISIT(t->backend);
  Py_VISIT(t->base);
  Py_VISIT(t->dict);
  return 0;
}
int tensor_clear(PyObject* self) {
  Tensor* t = reinterpret_cast<Tensor*>(self);
  Py_CLEAR(t->base);
  Py_CLEAR(t->dict);
  PyObject* backend = t->backend;
  Py_INCREF(Py_None);
  t->backend = Py_None;
  Py_XDECREF(backend);
  return 0;
}

PyObject* tensor_shape(PyObject* self, void*) {
  PyObject* shape = reinterpret_cast<Tensor*>(self)->shape;
  Py_INCREF(shape);
  return shape;
}
int tensor_set_shape(PyObject* self, PyObject* given, void*) {
  Tensor* t = reinterpret_cast<Tensor*>(self);
  PyObject* shape = given ? shape_tuple(given) : nullptr;
  if (!shape) {
    if (!given) PyErr_SetString(PyExc_AttributeError, "shape");
    return -1;
  }
  const Py_ssize_t n = elements(shape);
  if (n == -1 && PyErr_Occurred()) {
    Py_DECREF(shape);
    return -1;
  }
  t->numel = n;
  PyObject* old = t->shape;
  t->shape = shape;
  Py_DECREF(old);
  return 0;
}

PyObject* tensor_nbytes(PyObject* self, void*) {
  const Tensor* t = reinterpret_cast<const Tensor*>(self);
  return PyLong_FromSsize_t(t->numel * ((t->dtype >= 0 && t->dtype < 4) ? kSizes[t->dtype] : 0));
}

// reshape(*shape) or reshape(shape): a zero-copy view (tensor.rs:1555-1605) that does not own the memory.
PyObject* tensor_reshape(PyObject* self, PyObject* args) {
  Tensor* t = reinterpret_cast<Tensor*>(self);
  PyObject* given = args;
  if (PyTuple_GET_SIZE(args) == 1 && (PyTuple_Check(PyTuple_GET_ITEM(args, 0)) || PyList_Check(PyTuple_GET_ITEM(args, 0))))
    given = PyTuple_GET_ITEM(args, 0);
  PyObject* shape = shape_tuple(given);
  if (!shape) return nullptr;
  const Py_ssize_t n = elements(shape);
  if (n != t->numel) {
    if (!PyErr_Occurred()) {
      PyObject* text = PyUnicode_FromFormat("reshape %R -> %R", t->shape, shape);
      if (text) raise_text(OMX_SHAPE, PyUnicode_AsUTF8(text));
      Py_XDECREF(text);
    }
    Py_DECREF(shape);
    return nullptr;
  }
  Tensor* view = make_tensor(t->backend, t->context, t->ptr, shape, n, t->dtype, false);
  if (!view) return nullptr;
  Py_INCREF(self);
  view->base = self;
  view->compute_bf16 = t->compute_bf16;
  return reinterpret_cast<PyObject*>(view);
}

PyMethodDef tensor_methods[] = {{"reshape", tensor_reshape, METH_VARARGS, "A zero-copy view of another shape."},
                                {nullptr, nullptr, 0, nullptr}};
PyMemberDef tensor_members[] = {
    {"backend", T_OBJECT, offsetof(Tensor, backend), READONLY, nullptr},
    {"ptr", T_ULONGLONG, offsetof(Tensor, ptr), 0, nullptr},
    {"dtype", T_INT, offsetof(Tensor, dtype), 0, nullptr},
    {"numel", T_PYSSIZET, offsetof(Tensor, numel), READONLY, nullptr},
    {"_owns", T_BOOL, offsetof(Tensor, owns), 0, nullptr},
    {"_base", T_OBJECT, offsetof(Tensor, base), READONLY, nullptr},
    // The storage compute tag of an f32 tensor (tensor.rs COMPUTE_BF16): true when its values are known
    // to be bf16-exact, so a second rounding would only clone. Set by `Autocast`.
    {"compute_bf16", T_BOOL, offsetof(Tensor, compute_bf16), 0, nullptr},
    {nullptr, 0, 0, 0, nullptr}};
PyGetSetDef tensor_getset[] = {{"shape", tensor_shape, tensor_set_shape, nullptr, nullptr},
                               {"__dict__", PyObject_GenericGetDict, PyObject_GenericSetDict, nullptr, nullptr},
                               {"nbytes", tensor_nbytes, nullptr, nullptr, nullptr}, {nullptr, nullptr, nullptr, nullptr, nullptr}};

// empty(backend, context, shape, dtype): a new tensor charged to the context's budget.
PyObject* empty(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 4 || Py_TYPE(args[1]) != &ContextType) {
    PyErr_SetString(PyExc_TypeError, "empty(backend, context, shape, dtype)");
    return nullptr;
  }
  Context* c = reinterpret_cast<Context*>(args[1]);
  const long dtype = PyLong_AsLong(args[3]);
  if (dtype == -1 && PyErr_Occurred()) return nullptr;
  if (dtype < 0 || dtype > 3) {
    PyErr_SetObject(PyExc_KeyError, args[3]);
    return nullptr;
  }
  PyObject* shape = shape_tuple(args[2]);
  if (!shape) return nullptr;
  const Py_ssize_t n = elements(shape);
  if (n == -1 && PyErr_Occurred()) {
    Py_DECREF(shape);
    return nullptr;
  }
  void* p = nullptr;
  const int32_t rc = c->ctx && p_alloc ? p_alloc(c->ctx, static_cast<uint64_t>(n > 1 ? n : 1) * kSizes[dtype], &p) : OMX_BACKEND;
  if (rc != OMX_OK) {
    Py_DECREF(shape);
    return raise(c->ctx, rc);
  }
  Tensor* t = make_tensor(args[0], c, reinterpret_cast<unsigned long long>(p), shape, n, static_cast<int>(dtype), true);
  if (!t) p_free(c->ctx, p);
  return reinterpret_cast<PyObject*>(t);
}

// lists_match(list, list, ...), of one length: whether every entry's tensors are f32, have elements and share a shape. Returns
// their rank (0 where entries differ in it), or -1.
PyObject* lists_match(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs < 1) return PyLong_FromLong(-1);
  Py_ssize_t rank = -1;
  for (Py_ssize_t l = 0; l < nargs; ++l)
    if (!PyList_CheckExact(args[l]) || PyList_GET_SIZE(args[l]) != PyList_GET_SIZE(args[0])) return PyLong_FromLong(-1);
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(args[0]); ++i) {
    PyObject* first = nullptr;
    for (Py_ssize_t l = 0; l < nargs; ++l) {
      PyObject* o = PyList_GET_ITEM(args[l], i);
      if (Py_TYPE(o) != &TensorType) return PyLong_FromLong(-1);
      const Tensor* t = reinterpret_cast<const Tensor*>(o);
      if (t->dtype != 0 || t->numel <= 0) return PyLong_FromLong(-1);
      if (!first) first = t->shape;
      const int same = first == t->shape ? 1 : PyObject_RichCompareBool(first, t->shape, Py_EQ);
      if (same < 0) return nullptr;
      if (!same) return PyLong_FromLong(-1);
    }
    const Py_ssize_t own = PyTuple_GET_SIZE(first);
    rank = rank == -1 || rank == own ? own : 0;
  }
  return PyLong_FromSsize_t(rank);
}

// ---- typed calls ----
// One argument converted into parameter type T. A pointer is a tensor's memory, null or a plain
// address; a host array is refused (its address would reach a kernel).
template <typename T>
bool convert(PyObject* o, T* out) {
  if constexpr (std::is_same_v<T, omx_ctx*>) {
    if (Py_TYPE(o) != &ContextType) {
      PyErr_SetString(PyExc_TypeError, "the first argument is the backend's context");
      return false;
    }
    *out = reinterpret_cast<Context*>(o)->ctx;
    return true;
  } else if constexpr (std::is_pointer_v<T>) {
    if (PyObject_TypeCheck(o, &TensorType)) {
      *out = reinterpret_cast<T>(reinterpret_cast<Tensor*>(o)->ptr);
      return true;
    }
    if (o == Py_None) {
      *out = nullptr;
      return true;
    }
    if (PyLong_Check(o)) {
      const unsigned long long v = PyLong_AsUnsignedLongLong(o);
      *out = reinterpret_cast<T>(v);
      return !(v == static_cast<unsigned long long>(-1) && PyErr_Occurred());
    }
    if (std::is_same_v<T, const char*> && PyBytes_Check(o)) {
      *out = reinterpret_cast<T>(PyBytes_AS_STRING(o));
      return true;
    }
    PyErr_Format(PyExc_TypeError, "a device tensor is expected, not %.80s", Py_TYPE(o)->tp_name);
    return false;
  } else if constexpr (std::is_floating_point_v<T>) {
    const double v = PyFloat_AsDouble(o);
    *out = static_cast<T>(v);
    return !(v == -1.0 && PyErr_Occurred());
  } else if constexpr (std::is_signed_v<T>) {
    const long long v = PyLong_AsLongLong(o);
    *out = static_cast<T>(v);
    if (v == -1 && PyErr_Occurred()) return false;
    if (static_cast<long long>(*out) != v) {
      PyErr_SetString(PyExc_OverflowError, "argument out of range");
      return false;
    }
    return true;
  } else {
    PyObject* whole = PyNumber_Index(o);
    if (!whole) return false;
    const unsigned long long v = PyLong_AsUnsignedLongLong(whole);
    Py_DECREF(whole);
    *out = static_cast<T>(v);
    if (v == static_cast<unsigned long long>(-1) && PyErr_Occurred()) return false;
    if (static_cast<unsigned long long>(*out) != v) {
      PyErr_SetString(PyExc_OverflowError, "argument out of range");
      return false;
    }
    return true;
  }
}

// Entry<ID, Signature>: the function's address (filled by `load`) and the Python callable around it.
template <int ID, typename F>
struct Entry;
template <int ID, typename... P>
struct Entry<ID, int32_t(P...)> {
  static inline int32_t (*address)(P...) = nullptr;

  template <size_t... I>
  static PyObject* invoke(PyObject* const* args, std::index_sequence<I...>) {
    std::tuple<P...> v;
    if (!(convert(args[I], &std::get<I>(v)) && ...)) return nullptr;
    int32_t rc;
    Py_BEGIN_ALLOW_THREADS
    rc = address(std::get<I>(v)...);
    Py_END_ALLOW_THREADS
    if (rc != OMX_OK) return raise(std::get<0>(v), rc);
    Py_RETURN_NONE;
  }
  static PyObject* call(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    if (nargs != static_cast<Py_ssize_t>(sizeof...(P)) || !address) {
      PyErr_Format(PyExc_TypeError, address ? "%zu arguments expected" : "the library is not loaded", sizeof...(P));
      return nullptr;
    }
    return invoke(args, std::make_index_sequence<sizeof...(P)>{});
  }
};

struct Symbol {
  const char* name;
  void** address;
};

#define OMX_ENTRIES(X)                                                                                                   \
  X(omx_fill_zero) X(omx_upload) X(omx_upload_staged) X(omx_download) X(omx_sync) X(omx_cast_bf16) X(omx_to_bf16) X(omx_to_f32)               \
  X(omx_linear_forward) X(omx_linear_backward) X(omx_linear_backward_onto) X(omx_gemm) X(omx_gemm_strided_batch) X(omx_gemm_pitched_strided_batch)   \
  X(omx_linear_i8_group_forward) X(omx_linear_i8_group_backward_input) X(omx_pack_i8_group)                              \
  X(omx_causal_sdpa_forward) X(omx_causal_sdpa_backward) X(omx_causal_sdpa_backward_recompute)                           \
  X(omx_linear_gelu_forward) X(omx_linear_backward_input_gelu) X(omx_causal_attention_forward)                           \
  X(omx_causal_attention_backward) X(omx_causal_attention_f32_forward) X(omx_causal_attention_f32_backward) X(omx_causal_attention_forward_saving) X(omx_causal_attention_backward_saved)         \
  X(omx_rms_norm_forward) X(omx_rms_norm_backward) X(omx_residual_add_rms_norm_forward)                                  \
  X(omx_rms_norm_backward_residual) X(omx_cross_entropy_mean_forward) X(omx_cross_entropy_mean_forward_static)           \
  X(omx_cross_entropy_mean_backward) X(omx_linear_cross_entropy_mean) X(omx_embedding_forward) X(omx_embedding_backward) \
  X(omx_embedding_backward_accumulate) X(omx_adamw_step) X(omx_adamw_step_bounded) X(omx_muon_ns5_step)                  \
  X(omx_muon_ns5_step_batched) X(omx_muon_ns5_step_list) X(omx_muon_ns5_step_shapes) X(omx_adamw_step_batched) X(omx_accumulate_grads) X(omx_clip_grad_norm) X(omx_residual_add) X(omx_accumulate_grad) X(omx_scale_grad)        \
  X(omx_gelu_forward) X(omx_gelu_backward) X(omx_cached_attention_forward) X(omx_kv_cache_write) X(omx_token_windows)    \
  X(omx_permute_0213) X(omx_silu_forward) X(omx_silu_backward) X(omx_mul_forward) X(omx_mul_backward) X(omx_silu_mul_forward) X(omx_silu_mul_backward)                    \
  X(omx_rope_half_split_forward) X(omx_rope_half_split_backward) X(omx_rope_half_split_inplace)                          \
  X(omx_rope_half_split_pitched) X(omx_swiglu_forward) X(omx_swiglu_backward) X(omx_linear_swiglu_forward) X(omx_linear_i8_group_swiglu_forward) X(omx_linear_backward_input_swiglu) X(omx_linear_i8_group_backward_input_swiglu) X(omx_linear_i8_group_rope_forward) X(omx_rms_qk_norm_forward)                 \
  X(omx_rms_qk_norm_backward) X(omx_per_head_sigmoid_gate_forward) X(omx_per_head_sigmoid_gate_backward)                 \
  X(omx_per_head_sigmoid_gate_backward_deferred) X(omx_per_head_sigmoid_gate_sum_forward) X(omx_per_head_sigmoid_gate_sum_backward) X(omx_per_head_sigmoid_gate_input_grad_add)                             \
  X(omx_value_residual_blend_forward) X(omx_value_residual_blend_backward) X(omx_qkv_prepare_forward)                    \
  X(omx_qkv_prepare_backward) X(omx_argmax_rows) X(omx_topk_rows) X(omx_set_option)

enum EntryId {
#define X(name) ID_##name,
  OMX_ENTRIES(X)
#undef X
};
#define X(name) {#name, reinterpret_cast<void**>(&Entry<ID_##name, decltype(::name)>::address)},
Symbol g_symbols[] = {OMX_ENTRIES(X)};
#undef X

// ---- the backend's methods that a decoding loop calls for every token ----
// `MiBackend` derives from a type with these methods. Each takes the well-formed call from Python's arguments to the
// library's entry point; anything else (an operand that is no device tensor, a shape or dtype that does not fit, an
// unknown keyword) goes to the Python method of the same name behind `_checked_`, which says what is wrong. With the
// checks in Python a call of a 3 us launch spent 2 us on them: one token through 12 layers, 150 calls, 731 us; with
// these methods 551 us of host time, and the device is what bounds it.
struct Held {  // a new reference, dropped at the end of the scope
  PyObject* o;
  ~Held() { Py_XDECREF(o); }
};

PyObject* new_reference(PyObject* o) {
  Py_INCREF(o);
  return o;
}

// Positional and keyword arguments into `slot`, absent ones null; false where the names do not fit.
template <size_t N>
bool bind(PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames, const char* const (&names)[N], PyObject* (&slot)[N]) {
  if (nargs > static_cast<Py_ssize_t>(N)) return false;
  for (size_t i = 0; i < N; ++i) slot[i] = static_cast<Py_ssize_t>(i) < nargs ? args[i] : nullptr;
  const Py_ssize_t words = kwnames ? PyTuple_GET_SIZE(kwnames) : 0;
  for (Py_ssize_t w = 0; w < words; ++w) {
    size_t i = 0;
    while (i < N && PyUnicode_CompareWithASCIIString(PyTuple_GET_ITEM(kwnames, w), names[i]) != 0) ++i;
    if (i == N || slot[i]) return false;
    slot[i] = args[nargs + w];
  }
  return true;
}

const Tensor* tensor_in(PyObject* o) { return o && PyObject_TypeCheck(o, &TensorType) ? reinterpret_cast<const Tensor*>(o) : nullptr; }
// A float tensor with elements, as the validators ask of every operand.
const Tensor* floats_in(PyObject* o) {
  const Tensor* t = tensor_in(o);
  return t && (t->dtype == 0 || t->dtype == 1) && t->numel > 0 ? t : nullptr;
}
Py_ssize_t rank(const Tensor* t) { return PyTuple_GET_SIZE(t->shape); }
Py_ssize_t axis(const Tensor* t, Py_ssize_t i) { return PyLong_AsSsize_t(PyTuple_GET_ITEM(t->shape, i)); }
Py_ssize_t last_axis(const Tensor* t) { return axis(t, rank(t) - 1); }
// An optional dtype (None and absent: `otherwise`), -1 where it is none.
int dtype_in(PyObject* o, int otherwise) {
  if (!o || o == Py_None) return otherwise;
  if (!PyLong_CheckExact(o)) return -1;
  const long v = PyLong_AsLong(o);
  if (v == -1 && PyErr_Occurred()) PyErr_Clear();
  return v >= 0 && v <= 3 ? static_cast<int>(v) : -1;
}
// A whole number from 0 to 2^62, -1 where it is none.
long long count_in(PyObject* o) {
  if (!o || !PyLong_CheckExact(o)) return -1;
  const long long v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) PyErr_Clear();
  return v >= 0 && v <= (1ll << 62) ? v : -1;
}

PyObject* new_tensor(PyObject* backend, Context* c, PyObject* shape /* stolen */, int dtype) {
  if (!shape) return nullptr;
  const Py_ssize_t n = elements(shape);
  void* p = nullptr;
  const int32_t rc = c->ctx ? p_alloc(c->ctx, static_cast<uint64_t>(n > 1 ? n : 1) * kSizes[dtype], &p) : OMX_BACKEND;
  if (rc != OMX_OK) {
    Py_DECREF(shape);
    return raise(c->ctx, rc);
  }
  Tensor* t = make_tensor(backend, c, reinterpret_cast<unsigned long long>(p), shape, n, dtype, true);
  if (!t) p_free(c->ctx, p);
  return reinterpret_cast<PyObject*>(t);
}
// x's shape with its last axis (or, with `append`, one more axis) of `n`.
PyObject* shape_with(const Tensor* x, Py_ssize_t n, bool append) {
  const Py_ssize_t lead = rank(x) - (append ? 0 : 1);
  PyObject* shape = PyTuple_New(lead + 1);
  if (!shape) return nullptr;
  for (Py_ssize_t i = 0; i < lead; ++i) {
    PyObject* a = PyTuple_GET_ITEM(x->shape, i);
    Py_INCREF(a);
    PyTuple_SET_ITEM(shape, i, a);
  }
  PyObject* a = PyLong_FromSsize_t(n);
  if (!a) {
    Py_DECREF(shape);
    return nullptr;
  }
  PyTuple_SET_ITEM(shape, lead, a);
  return shape;
}
PyObject* shape_of(const Tensor* x) {
  Py_INCREF(x->shape);
  return x->shape;
}
template <typename T = void>
T* memory(const Tensor* t) {
  return reinterpret_cast<T*>(t->ptr);
}
template <typename T = void>
T* memory(const Held& h) {
  return reinterpret_cast<T*>(reinterpret_cast<const Tensor*>(h.o)->ptr);
}

// The call's context (a reference) and, where the fast path does not apply, its Python method.
Context* context_of(PyObject* self) {
  static PyObject* name = PyUnicode_InternFromString("_context");
  PyObject* c = PyObject_GetAttr(self, name);
  if (c && Py_TYPE(c) != &ContextType) Py_CLEAR(c);
  if (!c) PyErr_Clear();
  return reinterpret_cast<Context*>(c);
}
PyObject* in_python(PyObject* self, PyObject* name, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames) {
  Held method{PyObject_GetAttr(self, name)};
  return method.o ? PyObject_Vectorcall(method.o, args, nargs, kwnames) : nullptr;
}
// The library call without the interpreter lock; null with the error set where it refuses.
template <typename F>
bool without_lock(Context* c, F&& call) {
  int32_t rc;
  Py_BEGIN_ALLOW_THREADS
  rc = call(c->ctx);
  Py_END_ALLOW_THREADS
  if (rc != OMX_OK) raise(c->ctx, rc);
  return rc == OMX_OK;
}

#define OMX_METHOD(name) PyObject* m_##name(PyObject* self, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames)
#define OMX_IN_PYTHON(name)                                                 \
  do {                                                                      \
    static PyObject* checked = PyUnicode_InternFromString("_checked_" #name); \
    return in_python(self, checked, args, nargs, kwnames);                  \
  } while (0)
#define OMX_CALL(name) (reinterpret_cast<decltype(&::name)>(*g_symbols[ID_##name].address))

OMX_METHOD(linear_forward) {
  static const char* const names[] = {"x", "w", "out_dtype"};
  PyObject* slot[3];
  const bool bound = bind(args, nargs, kwnames, names, slot);
  const Tensor *x = bound ? floats_in(slot[0]) : nullptr, *w = bound ? floats_in(slot[1]) : nullptr;
  const int dtype = bound ? dtype_in(slot[2], 0) : -1;
  Held ctx{x && w ? reinterpret_cast<PyObject*>(context_of(self)) : nullptr};
  if (!ctx.o || dtype < 0 || rank(x) < 1 || rank(w) != 2 || last_axis(x) != axis(w, 1)) OMX_IN_PYTHON(linear_forward);
  Context* c = reinterpret_cast<Context*>(ctx.o);
  const Py_ssize_t kin = axis(w, 1), nout = axis(w, 0);
  Held y{new_tensor(self, c, shape_with(x, nout, false), dtype)};
  if (!y.o || !without_lock(c, [&](omx_ctx* o) {
        return OMX_CALL(omx_linear_forward)(o, memory(x), x->dtype, memory(w), w->dtype, memory(y), dtype, x->numel / kin, kin, nout);
      }))
    return nullptr;
  return new_reference(y.o);
}

OMX_METHOD(linear_gelu_forward) {
  static const char* const names[] = {"x", "w", "tanh_form"};
  PyObject* slot[3];
  const bool bound = bind(args, nargs, kwnames, names, slot);
  const Tensor *x = bound ? floats_in(slot[0]) : nullptr, *w = bound ? floats_in(slot[1]) : nullptr;
  Held ctx{x && w ? reinterpret_cast<PyObject*>(context_of(self)) : nullptr};
  if (!ctx.o || rank(x) < 1 || rank(w) != 2 || last_axis(x) != axis(w, 1) || (slot[2] && !PyBool_Check(slot[2])))
    OMX_IN_PYTHON(linear_gelu_forward);
  Context* c = reinterpret_cast<Context*>(ctx.o);
  const Py_ssize_t kin = axis(w, 1), nout = axis(w, 0);
  Held u{new_tensor(self, c, shape_with(x, nout, false), 1)};
  Held act{u.o ? new_tensor(self, c, shape_with(x, nout, false), 1) : nullptr};
  if (!act.o || !without_lock(c, [&](omx_ctx* o) {
        return OMX_CALL(omx_linear_gelu_forward)(o, memory(x), memory(w), x->dtype, memory(u), memory(act), x->numel / kin, kin, nout,
                                                 slot[2] == Py_True);
      }))
    return nullptr;
  return PyTuple_Pack(2, u.o, act.o);
}

OMX_METHOD(residual_add_rms_norm_forward) {
  static const char* const names[] = {"x", "y", "w", "eps", "out_dtype"};
  PyObject* slot[5];
  const bool bound = bind(args, nargs, kwnames, names, slot);
  const Tensor *x = bound ? floats_in(slot[0]) : nullptr, *y = bound ? floats_in(slot[1]) : nullptr;
  const Tensor* w = bound ? floats_in(slot[2]) : nullptr;
  const int dtype = y ? dtype_in(slot[4], y->dtype) : -1;
  Held ctx{x && y && w ? reinterpret_cast<PyObject*>(context_of(self)) : nullptr};
  if (!ctx.o || dtype < 0 || rank(x) < 1 || (slot[3] && !PyFloat_CheckExact(slot[3]))) OMX_IN_PYTHON(residual_add_rms_norm_forward);
  Context* c = reinterpret_cast<Context*>(ctx.o);
  const Py_ssize_t dim = last_axis(x);
  const float eps = slot[3] ? static_cast<float>(PyFloat_AS_DOUBLE(slot[3])) : 1e-6f;
  Held total{new_tensor(self, c, shape_of(x), 0)};
  Held normed{total.o ? new_tensor(self, c, shape_of(x), dtype) : nullptr};
  if (!normed.o || !without_lock(c, [&](omx_ctx* o) {
        return OMX_CALL(omx_residual_add_rms_norm_forward)(o, memory(x), x->dtype, memory(y), y->dtype, memory<float>(w), memory<float>(total),
                                                           memory(normed), dtype, x->numel / dim, dim, eps);
      }))
    return nullptr;
  return PyTuple_Pack(2, total.o, normed.o);
}

OMX_METHOD(to_bf16) {
  static const char* const names[] = {"x"};
  PyObject* slot[1];
  const Tensor* x = bind(args, nargs, kwnames, names, slot) ? floats_in(slot[0]) : nullptr;
  Held ctx{x ? reinterpret_cast<PyObject*>(context_of(self)) : nullptr};
  if (!ctx.o) OMX_IN_PYTHON(to_bf16);
  Context* c = reinterpret_cast<Context*>(ctx.o);
  Held y{new_tensor(self, c, shape_of(x), 1)};
  if (!y.o || !without_lock(c, [&](omx_ctx* o) { return OMX_CALL(omx_to_bf16)(o, memory<float>(x), memory(y), x->numel); })) return nullptr;
  return new_reference(y.o);
}

OMX_METHOD(embedding_forward) {
  static const char* const names[] = {"table", "ids", "out_dtype"};
  PyObject* slot[3];
  const bool bound = bind(args, nargs, kwnames, names, slot);
  const Tensor *table = bound ? floats_in(slot[0]) : nullptr, *ids = bound ? tensor_in(slot[1]) : nullptr;
  const int dtype = bound ? dtype_in(slot[2], 0) : -1;
  Held ctx{table && ids ? reinterpret_cast<PyObject*>(context_of(self)) : nullptr};
  if (!ctx.o || dtype < 0 || rank(table) != 2 || ids->dtype != 2 || ids->numel < 1) OMX_IN_PYTHON(embedding_forward);
  Context* c = reinterpret_cast<Context*>(ctx.o);
  const Py_ssize_t vocab = axis(table, 0), dim = axis(table, 1);
  Held y{new_tensor(self, c, shape_with(ids, dim, true), dtype)};
  if (!y.o || !without_lock(c, [&](omx_ctx* o) {
        return OMX_CALL(omx_embedding_forward)(o, memory(table), table->dtype, memory(ids), memory(y), dtype, ids->numel, vocab, dim);
      }))
    return nullptr;
  return new_reference(y.o);
}

OMX_METHOD(kv_cache_write) {
  static const char* const names[] = {"cache", "src", "at"};
  PyObject* slot[3];
  const bool bound = bind(args, nargs, kwnames, names, slot);
  const Tensor *cache = bound ? floats_in(slot[0]) : nullptr, *src = bound ? floats_in(slot[1]) : nullptr;
  const long long at = bound ? count_in(slot[2]) : -1;
  Held ctx{cache && src ? reinterpret_cast<PyObject*>(context_of(self)) : nullptr};
  if (!ctx.o || at < 0 || rank(cache) != 4 || rank(src) != 4 || src->dtype != 0 || axis(src, 0) != axis(cache, 0) ||
      axis(src, 2) != axis(cache, 2) || axis(src, 3) != axis(cache, 3) || axis(src, 1) > axis(cache, 1))
    OMX_IN_PYTHON(kv_cache_write);
  Context* c = reinterpret_cast<Context*>(ctx.o);
  if (!without_lock(c, [&](omx_ctx* o) {
        return OMX_CALL(omx_kv_cache_write)(o, memory(cache), cache->dtype, memory<float>(src), axis(cache, 0), axis(cache, 1), axis(cache, 2),
                                            axis(cache, 3), axis(src, 1), at);
      }))
    return nullptr;
  Py_RETURN_NONE;
}

OMX_METHOD(cached_attention_forward) {
  static const char* const names[] = {"q", "k_cache", "v_cache", "kv_len", "window"};
  PyObject* slot[5];
  const bool bound = bind(args, nargs, kwnames, names, slot);
  const Tensor *q = bound ? floats_in(slot[0]) : nullptr, *k = bound ? floats_in(slot[1]) : nullptr;
  const Tensor* v = bound ? floats_in(slot[2]) : nullptr;
  const long long kv_len = bound ? count_in(slot[3]) : -1;
  const long long window = bound && slot[4] && slot[4] != Py_None ? count_in(slot[4]) : 0;
  Held ctx{q && k && v ? reinterpret_cast<PyObject*>(context_of(self)) : nullptr};
  if (!ctx.o || kv_len < 0 || window < 0 || (slot[4] && slot[4] != Py_None && window == 0) || rank(q) != 4 || rank(k) != 4 ||
      rank(v) != 4 || q->dtype != 0 || k->dtype != v->dtype)
    OMX_IN_PYTHON(cached_attention_forward);
  const Py_ssize_t b = axis(q, 0), tq = axis(q, 1), h = axis(q, 2), d = axis(q, 3), cap = axis(k, 1), hkv = axis(k, 2);
  const long long span = window && window < kv_len && tq + window - 1 < kv_len ? tq + window - 1 : kv_len;
  bool fits = axis(k, 0) == b && axis(k, 3) == d && h % hkv == 0 && kv_len >= tq && span <= cap;
  for (Py_ssize_t i = 0; i < 4; ++i) fits &= axis(k, i) == axis(v, i);
  if (!fits) OMX_IN_PYTHON(cached_attention_forward);
  Context* c = reinterpret_cast<Context*>(ctx.o);
  Held out{new_tensor(self, c, shape_of(q), 0)};
  if (!out.o || !without_lock(c, [&](omx_ctx* o) {
        return OMX_CALL(omx_cached_attention_forward)(o, memory<float>(q), memory(k), memory(v), k->dtype, memory<float>(out), b, tq, h, hkv, d,
                                                      cap, kv_len, window);
      }))
    return nullptr;
  return new_reference(out.o);
}

#define OMX_METHODS(X)                                                                                              \
  X(linear_forward) X(linear_gelu_forward) X(residual_add_rms_norm_forward) X(to_bf16) X(embedding_forward)        \
  X(kv_cache_write) X(cached_attention_forward)
#define X(name) \
  {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&m_##name)), METH_FASTCALL | METH_KEYWORDS, "See `_checked_" #name "`."},
PyMethodDef backend_methods[] = {OMX_METHODS(X){nullptr, nullptr, 0, nullptr}};
#undef X
PyTypeObject MethodsType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// load(path, error_type): opens the library and finds every entry point.
PyObject* load(PyObject*, PyObject* args) {
  const char* path;
  PyObject* error;
  if (!PyArg_ParseTuple(args, "sO", &path, &error)) return nullptr;
  Py_INCREF(error);
  Py_XDECREF(g_error);
  g_error = error;
  if (p_alloc) Py_RETURN_NONE;
  void* lib = dlopen(path, RTLD_NOW | RTLD_LOCAL);
  if (!lib) return raise_text(OMX_BACKEND, dlerror());
  auto find = [&](const char* name) {
    void* p = dlsym(lib, name);
    if (!p) raise_text(OMX_BACKEND, name);
    return p;
  };
  for (const Symbol& s : g_symbols)
    if (!(*s.address = find(s.name))) return nullptr;
  void* alloc = find("omx_alloc");
  if (!alloc || !(p_free = reinterpret_cast<decltype(p_free)>(find("omx_free"))) ||
      !(p_last_error = reinterpret_cast<decltype(p_last_error)>(find("omx_last_error"))))
    return nullptr;
  p_alloc = reinterpret_cast<decltype(p_alloc)>(alloc);
  Py_RETURN_NONE;
}

#define X(name) \
  {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&Entry<ID_##name, decltype(::name)>::call)), METH_FASTCALL, nullptr},
PyMethodDef module_methods[] = {
    OMX_ENTRIES(X){"load", load, METH_VARARGS, "load(path, error_type)"},
    {"lists_match", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&lists_match)), METH_FASTCALL, "lists_match(list, ...)"},
    {"empty", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&empty)), METH_FASTCALL, "empty(backend, context, shape, dtype)"},
    {nullptr, nullptr, 0, nullptr}};
#undef X
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", "Typed calls into libojas_mi355x and its device tensor.", -1, module_methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) {
  ContextType.tp_name = "ojas_amd._native.Context";
  ContextType.tp_basicsize = sizeof(Context);
  ContextType.tp_flags = Py_TPFLAGS_DEFAULT;
  ContextType.tp_new = context_new;
  ContextType.tp_methods = context_methods;
  TensorType.tp_name = "ojas_amd._native.DeviceTensor";
  TensorType.tp_doc =
      "A contiguous device tensor: pointer, shape, dtype. Frees itself on drop\n"
      "(the role of `Arc<dyn DeviceBuffer>` + `Reservation`, tensor.rs:146-163).";
  TensorType.tp_basicsize = sizeof(Tensor);
  TensorType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_GC | Py_TPFLAGS_BASETYPE;
  TensorType.tp_dictoffset = offsetof(Tensor, dict);
  TensorType.tp_weaklistoffset = offsetof(Tensor, weak);
  TensorType.tp_new = tensor_new;
  TensorType.tp_init = tensor_init;
  TensorType.tp_dealloc = tensor_dealloc;
  TensorType.tp_traverse = tensor_traverse;
  TensorType.tp_clear = tensor_clear;
  TensorType.tp_methods = tensor_methods;
  TensorType.tp_members = tensor_members;
  TensorType.tp_getset = tensor_getset;
  MethodsType.tp_name = "ojas_amd._native.Methods";
  MethodsType.tp_doc = "The native methods of the backend class that derives from it.";
  MethodsType.tp_basicsize = sizeof(PyObject);
  MethodsType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE;
  MethodsType.tp_new = PyType_GenericNew;
  MethodsType.tp_methods = backend_methods;
  if (PyType_Ready(&ContextType) < 0 || PyType_Ready(&TensorType) < 0 || PyType_Ready(&MethodsType) < 0) return nullptr;
  PyObject* m = PyModule_Create(&module);
  if (!m) return nullptr;
  Py_INCREF(&ContextType);
  Py_INCREF(&TensorType);
  Py_INCREF(&MethodsType);
  if (PyModule_AddObject(m, "Methods", reinterpret_cast<PyObject*>(&MethodsType)) < 0 ||
      PyModule_AddObject(m, "Context", reinterpret_cast<PyObject*>(&ContextType)) < 0 ||
      PyModule_AddObject(m, "DeviceTensor", reinterpret_cast<PyObject*>(&TensorType)) < 0)
    return nullptr;
  return m;
}
