// The calls a step is made of, from Python without ctypes: arrays as objects that own their DLArray, and one function for each operator symbol
// that takes such arrays, numbers, a stream and a profiler as they are.
//
// What bounds a step of small operators is the host that issues it.  Through ctypes an operator call cost 1.1 us before the library was
// entered and a new array 1.5 us (a pointer object, a shape, a byref, twelve attributes), of 2 us that the launch itself takes: Relu 3.3 us, the
// small Transformer's step 1.37 ms for 0.73 ms of kernels.  The types of the arguments come from c_runtime_api.h, the addresses from the
// library that _base.py has loaded.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstddef>
#include <cstdint>
#include <cstring>
#include <tuple>
#include <type_traits>
#include <utility>
#include <vector>

#include "../../../include/c_runtime_api.h"

namespace {

PyObject *g_rules = nullptr;       // the dict with MEMORY_MANAGE_RULE
PyObject *g_recording = nullptr;   // the dict with _recording_keeper
PyObject *g_handle_of = nullptr;   // address -> ctypes handle
PyObject *g_pointers = nullptr;    // the ctypes types that a pointer may be of
PyObject *g_context = nullptr;     // DLContext
PyObject *g_structure = nullptr;   // ctypes.Structure
PyObject *g_rule_name, *g_keeper_name, *g_take_name, *g_handle_name;

// ---------------------------------------------------------------- arrays
struct Array {
  PyObject_HEAD
  DLArray *raw;
  char auto_deleted, is_view;
  // the rest of what NDArray carries; null: not set, the getters know the defaults
  PyObject *handle, *owner, *keeper, *stensor, *events, *swap, *in_gpu, *splitted, *split_number, *split_dimension;
};
extern PyTypeObject ArrayType;

int (*fn_alloc)(const index_t *, index_t, DLContext, DLArrayHandle *, int) = nullptr;
int (*fn_free)(DLArrayHandle, int) = nullptr;

// the memory rule; false while the interpreter goes down, and with an error set where it is no whole number
bool current_rule(int &rule) {
  PyObject *r = g_rules ? PyDict_GetItem(g_rules, g_rule_name) : nullptr;
  if (!r || r == Py_None) return false;
  rule = static_cast<int>(PyLong_AsLong(r));
  return !(rule == -1 && PyErr_Occurred());
}

// the address a ctypes pointer holds
bool pointer_of(PyObject *p, void **out) {
  bool is = false;   // (PyObject_IsInstance would look for __instancecheck__ each time)
  for (Py_ssize_t i = 0; g_pointers && !is && i < PyTuple_GET_SIZE(g_pointers); ++i)
    is = PyObject_TypeCheck(p, reinterpret_cast<PyTypeObject *>(PyTuple_GET_ITEM(g_pointers, i)));
  if (!is) {
    PyErr_Format(PyExc_TypeError, "a pointer, not %R", p);
    return false;
  }
  Py_buffer b;
  if (PyObject_GetBuffer(p, &b, PyBUF_SIMPLE)) return false;
  const bool ok = b.len == static_cast<Py_ssize_t>(sizeof(void *));
  if (ok) *out = *static_cast<void **>(b.buf);
  PyBuffer_Release(&b);
  if (!ok) PyErr_SetString(PyExc_TypeError, "not a pointer");
  return ok;
}

// the array's DLArray (a pointer object that it was given may have been filled in since)
DLArray *raw_of(Array *a) {
  void *p = nullptr;
  if (!a->raw && a->handle && a->handle != Py_None) {
    if (pointer_of(a->handle, &p)) a->raw = static_cast<DLArray *>(p);
    PyErr_Clear();
  }
  return a->raw;
}

int array_traverse(Array *a, visitproc visit, void *arg) {
  Py_VISIT(a->handle);
  Py_VISIT(a->owner);
  Py_VISIT(a->keeper);
  Py_VISIT(a->stensor);
  Py_VISIT(a->events);
  Py_VISIT(a->swap);
  Py_VISIT(a->in_gpu);
  Py_VISIT(a->splitted);
  Py_VISIT(a->split_number);
  Py_VISIT(a->split_dimension);
  return 0;
}
// Gives the memory back, once.  A finalizer: it runs for every array of a collected cycle before anything of the cycle is cleared, a
// recording's keeper among it (a view's memory is its owner's, which may go first).
void array_finalize(Array *a) {
  PyObject *type, *value, *trace;
  PyErr_Fetch(&type, &value, &trace);
  DLArray *raw = raw_of(a);
  a->raw = nullptr;
  if (!raw) return PyErr_Restore(type, value, trace);
  int rule = 0;
  bool mine = true;
  if (!current_rule(rule)) {
    mine = false;
    if (PyErr_Occurred()) PyErr_WriteUnraisable(reinterpret_cast<PyObject *>(a));
  } else if (a->is_view) {
    raw->data = nullptr;   // a view owns its struct and shape but not its data
  } else if (!a->auto_deleted) {
    mine = false;
  } else if (a->keeper && a->keeper != Py_None && raw->ctx.device_type == kGPU) {
    // an array born inside a recorded step outlives this object: the graph replays into it
    PyObject *handle = a->handle && a->handle != Py_None ? (Py_INCREF(a->handle), a->handle)
                                                         : PyObject_CallFunction(g_handle_of, "n", reinterpret_cast<Py_ssize_t>(raw));
    PyObject *taken = handle ? PyObject_CallMethodObjArgs(a->keeper, g_take_name, handle, PyDict_GetItem(g_rules, g_rule_name), nullptr) : nullptr;
    if (!taken) PyErr_WriteUnraisable(a->keeper);
    mine = taken && !PyObject_IsTrue(taken);
    Py_XDECREF(taken);
    Py_XDECREF(handle);
  }
  if (mine) {
    Py_BEGIN_ALLOW_THREADS
    fn_free(raw, rule);
    Py_END_ALLOW_THREADS
  }
  Py_CLEAR(a->handle);
  PyErr_Restore(type, value, trace);
}
int array_clear(Array *a) {
  Py_CLEAR(a->handle);
  Py_CLEAR(a->owner);
  Py_CLEAR(a->keeper);
  Py_CLEAR(a->stensor);
  Py_CLEAR(a->events);
  Py_CLEAR(a->swap);
  Py_CLEAR(a->in_gpu);
  Py_CLEAR(a->splitted);
  Py_CLEAR(a->split_number);
  Py_CLEAR(a->split_dimension);
  return 0;
}
void array_dealloc(Array *a) {
  // (a subclass's own deallocation has run the finalizer)
  if (Py_TYPE(a) == &ArrayType && PyObject_CallFinalizerFromDealloc(reinterpret_cast<PyObject *>(a))) return;
  PyObject_GC_UnTrack(a);
  array_clear(a);
  Py_TYPE(a)->tp_free(reinterpret_cast<PyObject *>(a));
}

int array_init(Array *a, PyObject *args, PyObject *kwargs) {
  static const char *names[] = {"handle", "auto_deleted", "owner", "is_view", nullptr};
  PyObject *handle, *owner = Py_None;
  int auto_deleted = 1, is_view = 0;
  if (!PyArg_ParseTupleAndKeywords(args, kwargs, "O|pOp", const_cast<char **>(names), &handle, &auto_deleted, &owner, &is_view)) return -1;
  void *raw = nullptr;
  if (handle != Py_None && !pointer_of(handle, &raw)) return -1;
  a->raw = static_cast<DLArray *>(raw);
  a->auto_deleted = auto_deleted;
  a->is_view = is_view;
  Py_INCREF(handle);
  Py_XSETREF(a->handle, handle);
  Py_INCREF(owner);
  Py_XSETREF(a->owner, owner);
  PyObject *k = PyDict_GetItem(g_recording, g_keeper_name);
  Py_XINCREF(k);
  Py_XSETREF(a->keeper, k);
  return 0;
}

PyObject *get_handle(Array *a, void *) {
  if (!a->handle) {
    if (!a->raw) Py_RETURN_NONE;
    a->handle = PyObject_CallFunction(g_handle_of, "n", reinterpret_cast<Py_ssize_t>(a->raw));
    if (!a->handle) return nullptr;
  }
  Py_INCREF(a->handle);
  return a->handle;
}
int set_handle(Array *a, PyObject *v, void *) {
  void *raw = nullptr;
  if (!v) v = Py_None;
  if (v != Py_None && !pointer_of(v, &raw)) return -1;
  a->raw = static_cast<DLArray *>(raw);
  Py_INCREF(v);
  Py_XSETREF(a->handle, v);
  return 0;
}
PyObject *get_shape(Array *a, void *) {
  const DLArray *raw = raw_of(a);
  if (!raw) {
    PyErr_SetString(PyExc_AttributeError, "the array has no handle");
    return nullptr;
  }
  PyObject *t = PyTuple_New(raw->ndim);
  for (int i = 0; t && i < raw->ndim; ++i) PyTuple_SET_ITEM(t, i, PyLong_FromLongLong(raw->shape[i]));
  return t;
}
PyObject *get_data_ptr(Array *a, void *) {
  const DLArray *raw = raw_of(a);
  if (!raw || !raw->data) Py_RETURN_NONE;
  return PyLong_FromVoidPtr(raw->data);
}
// attributes with a default that is made when first read (a list, a dict) or is the same for all
enum Default { kNone, kFalse, kTrue, kOne, kList, kDict };
struct Field {
  size_t at;
  Default otherwise;
};
PyObject *get_field(Array *a, void *closure) {
  const Field &f = *static_cast<Field *>(closure);
  PyObject *&v = *reinterpret_cast<PyObject **>(reinterpret_cast<char *>(a) + f.at);
  if (!v) switch (f.otherwise) {
      case kNone: Py_RETURN_NONE;
      case kFalse: Py_RETURN_FALSE;
      case kTrue: Py_RETURN_TRUE;
      case kOne: return PyLong_FromLong(1);
      case kList: v = PyList_New(0); break;
      case kDict: v = PyDict_New(); break;
    }
  Py_XINCREF(v);
  return v;
}
int set_field(Array *a, PyObject *value, void *closure) {
  PyObject *&v = *reinterpret_cast<PyObject **>(reinterpret_cast<char *>(a) + static_cast<Field *>(closure)->at);
  Py_XINCREF(value);
  Py_XSETREF(v, value);
  return 0;
}
Field f_owner{offsetof(Array, owner), kNone}, f_keeper{offsetof(Array, keeper), kNone}, f_stensor{offsetof(Array, stensor), kList},
    f_events{offsetof(Array, events), kDict}, f_swap{offsetof(Array, swap), kFalse}, f_in_gpu{offsetof(Array, in_gpu), kTrue},
    f_splitted{offsetof(Array, splitted), kFalse}, f_number{offsetof(Array, split_number), kOne}, f_dimension{offsetof(Array, split_dimension), kNone};

PyObject *get_flag(Array *a, void *at) { return PyBool_FromLong(*(reinterpret_cast<char *>(a) + *static_cast<size_t *>(at))); }
int set_flag(Array *a, PyObject *value, void *at) {
  const int t = value ? PyObject_IsTrue(value) : 0;
  if (t >= 0) *(reinterpret_cast<char *>(a) + *static_cast<size_t *>(at)) = static_cast<char>(t);
  return t < 0 ? -1 : 0;
}
size_t at_auto_deleted = offsetof(Array, auto_deleted), at_is_view = offsetof(Array, is_view);

#define FIELD(name, f) {name, reinterpret_cast<getter>(get_field), reinterpret_cast<setter>(set_field), nullptr, &f}
PyGetSetDef array_getset[] = {{"handle", reinterpret_cast<getter>(get_handle), reinterpret_cast<setter>(set_handle), nullptr, nullptr},
                              {"shape", reinterpret_cast<getter>(get_shape), nullptr, nullptr, nullptr},
                              {"data_ptr", reinterpret_cast<getter>(get_data_ptr), nullptr, nullptr, nullptr},
                              {"auto_deleted", reinterpret_cast<getter>(get_flag), reinterpret_cast<setter>(set_flag), nullptr, &at_auto_deleted},
                              {"_is_view", reinterpret_cast<getter>(get_flag), reinterpret_cast<setter>(set_flag), nullptr, &at_is_view},
                              FIELD("_owner", f_owner),
                              FIELD("_keeper", f_keeper),
                              FIELD("sTensor", f_stensor),
                              FIELD("_events", f_events),
                              FIELD("swap", f_swap),
                              FIELD("in_gpu", f_in_gpu),
                              FIELD("splitted", f_splitted),
                              FIELD("split_number", f_number),
                              FIELD("split_dimension", f_dimension),
                              {nullptr, nullptr, nullptr, nullptr, nullptr}};

PyTypeObject ArrayType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// new_array(type, shape, ctx): an array of `type`, a subclass of Array
PyObject *new_array(PyObject *, PyObject *const *args, Py_ssize_t n) {
  if (n != 3 || !PyType_Check(args[0]) || !PyType_IsSubtype(reinterpret_cast<PyTypeObject *>(args[0]), &ArrayType)) {
    PyErr_SetString(PyExc_TypeError, "new_array(type, shape, ctx)");
    return nullptr;
  }
  int rule = 0;
  if (!fn_alloc || !current_rule(rule)) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, "the library is not bound");
    return nullptr;
  }
  if (!PyObject_TypeCheck(args[2], reinterpret_cast<PyTypeObject *>(g_context))) return PyErr_Format(PyExc_TypeError, "ctx is a DLContext, not %R", args[2]);
  Py_buffer b;
  if (PyObject_GetBuffer(args[2], &b, PyBUF_SIMPLE)) return nullptr;
  DLContext ctx{};
  const bool context = b.len == static_cast<Py_ssize_t>(sizeof ctx);
  if (context) ctx = *static_cast<DLContext *>(b.buf);
  PyBuffer_Release(&b);
  if (!context) {
    PyErr_SetString(PyExc_TypeError, "ctx is not a DLContext");
    return nullptr;
  }
  PyObject *seq = PySequence_Fast(args[1], "a shape is a sequence of whole numbers");
  if (!seq) return nullptr;
  const Py_ssize_t ndim = PySequence_Fast_GET_SIZE(seq);
  index_t few[8];
  std::vector<index_t> many(ndim > 8 ? ndim : 0);
  index_t *shape = ndim > 8 ? many.data() : few;
  bool ok = true;
  for (Py_ssize_t i = 0; ok && i < ndim; ++i) {
    PyObject *item = PySequence_Fast_GET_ITEM(seq, i), *whole = PyLong_Check(item) ? (Py_INCREF(item), item) : PyNumber_Long(item);
    shape[i] = whole ? PyLong_AsLongLong(whole) : -1;
    Py_XDECREF(whole);
    ok = !(shape[i] == -1 && PyErr_Occurred());
  }
  Py_DECREF(seq);
  if (!ok) return nullptr;
  PyTypeObject *type = reinterpret_cast<PyTypeObject *>(args[0]);
  Array *a = reinterpret_cast<Array *>(type->tp_alloc(type, 0));   // zeroed: every attribute has its default
  if (!a) return nullptr;
  a->auto_deleted = 1;
  PyObject *k = PyDict_GetItem(g_recording, g_keeper_name);
  if (k && k != Py_None) {
    Py_INCREF(k);
    a->keeper = k;
  }
  DLArrayHandle raw = nullptr;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = fn_alloc(shape, ndim, ctx, &raw, rule);
  Py_END_ALLOW_THREADS
  if (rc) {
    Py_DECREF(a);
    return PyErr_Format(PyExc_RuntimeError, "libc_runtime_api call failed with code %d", rc);
  }
  a->raw = raw;
  return reinterpret_cast<PyObject *>(a);
}

// ---------------------------------------------------------------- operator calls
template <class T>
struct Arg {   // whole numbers and truth values
  static bool get(PyObject *o, bool, T &v) {
    if constexpr (std::is_same<T, bool>::value) {
      const int t = PyObject_IsTrue(o);
      v = t > 0;
      return t >= 0;
    }
    // (as ctypes takes a size_t and int() an int)
    PyObject *whole = PyLong_Check(o) ? (Py_INCREF(o), o) : std::is_same<T, size_t>::value ? PyNumber_Index(o) : PyNumber_Long(o);
    if (!whole) return false;
    const unsigned long long bits = PyLong_AsUnsignedLongLongMask(whole);
    Py_DECREF(whole);
    v = static_cast<T>(bits);
    return !(bits == static_cast<unsigned long long>(-1) && PyErr_Occurred());
  }
};
template <>
struct Arg<float> {
  static bool get(PyObject *o, bool, float &v) {
    const double d = PyFloat_AsDouble(o);
    v = static_cast<float>(d);
    return !(d == -1.0 && PyErr_Occurred());
  }
};
template <>
struct Arg<DLArrayHandle> {
  static bool get(PyObject *o, bool optional, DLArrayHandle &v) {
    if (PyObject_TypeCheck(o, &ArrayType)) {
      v = raw_of(reinterpret_cast<Array *>(o));
      return true;
    }
    v = nullptr;
    if (optional) {
      const int given = PyObject_IsTrue(o);
      if (given <= 0) return given == 0;
    }
    PyErr_Format(PyExc_AssertionError, "an NDArray, not %R", o);
    return false;
  }
};
template <>
struct Arg<DLStreamHandle> {   // an object with a `handle`, or nothing: the default stream
  static bool get(PyObject *o, bool, DLStreamHandle &v) {
    v = nullptr;
    const int given = o == Py_None ? 0 : PyObject_IsTrue(o);
    if (given <= 0) return given == 0;
    PyObject *h = PyObject_GetAttr(o, g_handle_name);
    void *p = nullptr;
    const bool ok = h && (h == Py_None || pointer_of(h, &p));
    Py_XDECREF(h);
    v = static_cast<DLStreamHandle>(p);
    return ok;
  }
};
template <>
struct Arg<ProfilerHandle> {   // a Profiler structure or one that begins as it does, or nothing
  static bool get(PyObject *o, bool, ProfilerHandle &v) {
    v = nullptr;
    const int given = o == Py_None ? 0 : PyObject_IsTrue(o);
    if (given <= 0) return given == 0;
    Py_buffer b;
    const bool structure = PyObject_TypeCheck(o, reinterpret_cast<PyTypeObject *>(g_structure));
    if (!structure) PyErr_Format(PyExc_TypeError, "a Profiler, not %R", o);
    if (!structure || PyObject_GetBuffer(o, &b, PyBUF_WRITABLE)) return false;
    const bool ok = b.len >= static_cast<Py_ssize_t>(sizeof(Profiler));
    v = static_cast<ProfilerHandle>(b.buf);
    PyBuffer_Release(&b);   // the structure stays where it is: the caller holds it
    if (!ok) PyErr_SetString(PyExc_TypeError, "not a Profiler");
    return ok;
  }
};

template <class Op, class... A, size_t... I>
PyObject *call(int (*fn)(A...), PyObject *const *args, Py_ssize_t n, std::index_sequence<I...>) {
  if (n != static_cast<Py_ssize_t>(sizeof...(A))) return PyErr_Format(PyExc_TypeError, "%s takes %d arguments", Op::name(), static_cast<int>(sizeof...(A)));
  if (!fn) return PyErr_Format(PyExc_AttributeError, "the library has no %s", Op::name());
  std::tuple<A...> v;
  if (!(Arg<A>::get(args[I], Op::optional >> I & 1, std::get<I>(v)) && ...)) return nullptr;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = fn(std::get<I>(v)...);
  Py_END_ALLOW_THREADS
  if (rc) return PyErr_Format(PyExc_RuntimeError, "libc_runtime_api call failed with code %d", rc);
  Py_RETURN_NONE;
}
template <class Op, class... A>
PyObject *unpack(int (*fn)(A...), PyObject *const *args, Py_ssize_t n) {
  return call<Op>(fn, args, n, std::index_sequence_for<A...>{});
}
template <class Op>
PyObject *entry(PyObject *, PyObject *const *args, Py_ssize_t n) {
  return unpack<Op>(Op::fn, args, n);
}

// optional: a bit for every array argument that may be left out
#define CALLS(X)                                                                                                                              \
  X(DLGpuArraySet, 0) X(DLGpuMatrixElementwiseAdd, 0) X(DLGpuMatrixElementwiseAddByConst, 0) X(DLGpuMatrixElementwiseMultiply, 0)              \
  X(DLGpuMatrixMultiplyByConst, 0) X(DLGpuReshape, 0) X(DLGpuRelu, 0) X(DLGpuReluGradient, 0) X(DLGpuMatrixMultiply, 0)                        \
  X(TSplit_MatrixMultiplyAdd, 1 << 4 | 1 << 5 | 1 << 6 | 1 << 8) X(TSplit_MatrixMultiplySums, 0)                                               \
  X(TSplit_HeadsMatrixMultiply, 1 << 7 | 1 << 11) X(TSplit_HeadsScale, 0) X(DLGpuSoftmax, 0) X(DLGpuSoftmaxCrossEntropy, 0)                    \
  X(DLGpuSoftmaxCrossEntropy_Gradient, 0) X(TSplit_SoftmaxCrossEntropyIds, 0) X(TSplit_SoftmaxCrossEntropyIds_Gradient, 0)                     \
  X(TSplit_EmbeddingAdd, 0) X(TSplit_EmbeddingAdd_Gradient, 0) X(CuDNN_DLGpuConv2d, 0) X(CuDNN_DLGpuConv2d_Gradient_of_Filter, 0)              \
  X(CuDNN_DLGpuConv2d_Gradient_of_Data, 0) X(TSplit_Conv2dGradientOfDataAdd, 0) X(CuDNN_DLGpuBatch_Normalization, 1 << 6 | 1 << 7)              \
  X(CuDNN_DLGpuBatch_Normalization_gradient, 1 << 7 | 1 << 8) X(DLGpuMax_Pooling2d, 0) X(DLGpuMax_Pooling2d_gradient, 0)                       \
  X(CuDNN_DLGpuMax_Pooling2d, 0) X(CuDNN_DLGpuMax_Pooling2d_gradient, 0) X(SGDOptimizerUpdate, 0) X(MomentumOptimizerUpdate, 0)                \
  X(DLGpuAvgerage_Pooling2d, 0) X(DLGpuAvgerage_Pooling2d_gradient, 0) X(CuDNN_DLGpuAvgerage_Pooling2d, 0)                                     \
  X(CuDNN_DLGpuAvgerage_Pooling2d_gradient, 0) X(DLGpuBroadcastTo, 0) X(DLGpuReduceSumAxisZero, 0) X(DLGpuConv2d_broadcast_to, 0)              \
  X(DLGpuConv2d_reduce_sum, 0) X(DLGpuBatchMatrixMultiply, 0) X(DLGpuOneHot, 0) X(DLGpuWhere, 0) X(DLGpuEmbeddingLookUp, 0)                    \
  X(DLGpuEmbeddingLookUp_Gradient, 0) X(DLGpuTanh, 0) X(DLGpuSigmoid, 0) X(TSplit_BatchNormRelu, 0) X(TSplit_BatchNormReluAdd, 0)              \
  X(TSplit_BatchNormThenRelu, 1 << 7 | 1 << 8) X(TSplit_BatchNormThenRelu_gradient, 1 << 9 | 1 << 10) X(TSplit_Conv2dBatchNormStats, 0)        \
  X(TSplit_BatchNormFromStats, 1 << 7 | 1 << 8) X(TSplit_BatchNormRelu_gradient, 0) X(DLGpuConcat, 0) X(DLGpuConcat_gradient, 0)

#define DECLARE(symbol, mask)                                    \
  struct Op_##symbol {                                           \
    static const char *name() { return #symbol; }                \
    static constexpr unsigned optional = mask;                   \
    static inline decltype(&symbol) fn = nullptr;                \
  };
CALLS(DECLARE)

// bind(addresses by name, those of operators that the library lacks left out, the module dict with MEMORY_MANAGE_RULE, the one with
// _recording_keeper, address -> handle, the types of pointers, DLContext, ctypes.Structure)
PyObject *bind(PyObject *, PyObject *args) {
  PyObject *addresses, *rules, *recording, *handle_of, *pointers, *context, *structure;
  if (!PyArg_ParseTuple(args, "O!O!O!OO!O!O!", &PyDict_Type, &addresses, &PyDict_Type, &rules, &PyDict_Type, &recording, &handle_of, &PyTuple_Type,
                        &pointers, &PyType_Type, &context, &PyType_Type, &structure))
    return nullptr;
  auto look = [&](const char *name, auto &fn) {
    PyObject *a = PyDict_GetItemString(addresses, name);
    void *p = a ? PyLong_AsVoidPtr(a) : nullptr;
    fn = reinterpret_cast<typename std::remove_reference<decltype(fn)>::type>(p);
    return !PyErr_Occurred();
  };
#define BIND(symbol, mask) \
  if (!look(#symbol, Op_##symbol::fn)) return nullptr;
  CALLS(BIND)
  if (!look("DLArrayAlloc", fn_alloc) || !look("DLArrayFree", fn_free)) return nullptr;
  if (!fn_alloc || !fn_free) {
    PyErr_SetString(PyExc_AttributeError, "the library has no DLArrayAlloc or no DLArrayFree");
    return nullptr;
  }
  Py_INCREF(rules);
  Py_XSETREF(g_rules, rules);
  Py_INCREF(recording);
  Py_XSETREF(g_recording, recording);
  Py_INCREF(handle_of);
  Py_XSETREF(g_handle_of, handle_of);
  Py_INCREF(pointers);
  Py_XSETREF(g_pointers, pointers);
  Py_INCREF(context);
  Py_XSETREF(g_context, context);
  Py_INCREF(structure);
  Py_XSETREF(g_structure, structure);
  Py_RETURN_NONE;
}

#define METHOD(symbol, mask) {#symbol, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(entry<Op_##symbol>)), METH_FASTCALL, nullptr},
PyMethodDef methods[] = {CALLS(METHOD){"new_array", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(new_array)), METH_FASTCALL, nullptr},
                         {"bind", bind, METH_VARARGS, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__calls() {
  ArrayType.tp_name = "tsplit_amd._calls.Array";
  ArrayType.tp_basicsize = sizeof(Array);
  ArrayType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE | Py_TPFLAGS_HAVE_GC;
  ArrayType.tp_dealloc = reinterpret_cast<destructor>(array_dealloc);
  ArrayType.tp_traverse = reinterpret_cast<traverseproc>(array_traverse);
  ArrayType.tp_clear = reinterpret_cast<inquiry>(array_clear);
  ArrayType.tp_finalize = reinterpret_cast<destructor>(array_finalize);
  ArrayType.tp_init = reinterpret_cast<initproc>(array_init);
  ArrayType.tp_new = PyType_GenericNew;
  ArrayType.tp_getset = array_getset;
  if (PyType_Ready(&ArrayType)) return nullptr;
  g_rule_name = PyUnicode_InternFromString("MEMORY_MANAGE_RULE");
  g_keeper_name = PyUnicode_InternFromString("_recording_keeper");
  g_take_name = PyUnicode_InternFromString("take");
  g_handle_name = PyUnicode_InternFromString("handle");
  PyObject *m = PyModule_Create(&module);
  PyObject *names = PyList_New(0);
  if (!m || !names) return nullptr;
  for (const PyMethodDef *d = methods; d->ml_name; ++d)
    if (d->ml_flags == METH_FASTCALL && std::strcmp(d->ml_name, "new_array")) {
      PyObject *s = PyUnicode_FromString(d->ml_name);
      PyList_Append(names, s);
      Py_DECREF(s);
    }
  PyModule_AddObject(m, "SYMBOLS", names);
  Py_INCREF(&ArrayType);
  PyModule_AddObject(m, "Array", reinterpret_cast<PyObject *>(&ArrayType));
  return m;
}
