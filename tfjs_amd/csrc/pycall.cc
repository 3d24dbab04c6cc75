// The way from Python into the entry points that a program calls once per layer.
//
// ctypes converts every argument through a from_param() of its type: 0.75 us for the 16 arguments of tfhip_fused_matmul, and 0.35
// us for the call itself, where the launch takes 2.5 to 3.3. Here the argument types are the entry point's own, so the
// conversions are compiled: integers, None, floats and arrays of c_int64 are taken as they are. Whatever else
// an argument may be (c_void_p, byref(), a number out of range, a count that does not match) goes to the ctypes function, which decides
// as it always has. us per call on the host, ctypes and here: pyhost.device_fused_matmul 4.7 and 3.8, tfhip_fused_depthwise_conv2d 4.4
// and 3.7 (of the latter the launch itself is all but 0.3). Likewise the manifest of a weight buffer: 52 tensors took 24 us to read
// and 12 to wrap.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstddef>
#include <cstdint>
#include <cstring>
#include <limits>
#include <new>
#include <tuple>
#include <type_traits>
#include <utility>
#include <vector>

#include "tfjs_hip.h"

namespace {

PyObject *g_array_type = nullptr, *g_int64_type = nullptr;   // ctypes.Array, ctypes.c_int64
PyObject *g_underscore_type = nullptr;                       // "_type_"

// Types of c_int64 arrays that have been seen (there is one per length).
constexpr int kMaxTypes = 8;
PyTypeObject *g_types[kMaxTypes] = {};
int g_num_types = 0;

bool is_int64_array(PyObject *o) {
  PyTypeObject *type = Py_TYPE(o);
  for (int i = 0; i < g_num_types; ++i)
    if (g_types[i] == type) return true;
  if (!g_array_type || !PyType_IsSubtype(type, reinterpret_cast<PyTypeObject *>(g_array_type))) return false;
  PyObject *element = PyObject_GetAttr(reinterpret_cast<PyObject *>(type), g_underscore_type);
  const bool yes = element == g_int64_type;
  if (!element) PyErr_Clear();
  Py_XDECREF(element);
  if (yes && g_num_types < kMaxTypes) {
    Py_INCREF(type);
    g_types[g_num_types++] = type;
  }
  return yes;
}

// from(): whether the object has the form; the value is then in `to`.
bool from(PyObject *o, int64_t &to) {
  if (!PyLong_Check(o)) return false;
  int overflow = 0;
  to = PyLong_AsLongLongAndOverflow(o, &overflow);
  return overflow == 0;
}
bool from(PyObject *o, int &to) {
  int64_t v = 0;
  if (!from(o, v) || v < std::numeric_limits<int>::min() || v > std::numeric_limits<int>::max()) return false;
  to = (int)v;
  return true;
}
bool from(PyObject *o, double &to) {
  if (!PyFloat_CheckExact(o)) return false;
  to = PyFloat_AS_DOUBLE(o);
  return true;
}
bool from_address(PyObject *o, void *&to) {
  if (o == Py_None) {
    to = nullptr;
    return true;
  }
  int64_t v = 0;   // (an address in the upper half: ctypes)
  if (!from(o, v) || v < 0) return false;
  to = reinterpret_cast<void *>(static_cast<uintptr_t>(v));
  return true;
}
bool from(PyObject *o, const float *&to) {
  void *p = nullptr;
  if (!from_address(o, p)) return false;
  to = static_cast<const float *>(p);
  return true;
}
bool from(PyObject *o, void *&to) { return from_address(o, to); }
bool from(PyObject *, const void *&) { return false; }   // (of tfhip_decode_weights, called by position: ctypes)
bool from(PyObject *, void **&) { return false; }
bool from(PyObject *, const int *&) { return false; }
bool from(PyObject *, const double *&) { return false; }
bool from(PyObject *, size_t &) { return false; }
bool from(PyObject *o, float *&to) {
  void *p = nullptr;
  if (!from_address(o, p)) return false;
  to = static_cast<float *>(p);
  return true;
}
bool from(PyObject *o, const int64_t *&to) {
  if (o == Py_None) {
    to = nullptr;
    return true;
  }
  Py_buffer view;
  if (!is_int64_array(o)) return false;
  if (PyObject_GetBuffer(o, &view, PyBUF_SIMPLE) != 0) {
    PyErr_Clear();
    return false;
  }
  to = static_cast<const int64_t *>(view.buf);   // (the caller holds the array while the call lasts; it cannot be resized)
  PyBuffer_Release(&view);
  return true;
}

// ---- entry points by position

struct Entry {
  PyObject_HEAD
  vectorcallfunc call;
  PyObject *weak_references, *function;   // the ctypes function
  void *address;
};

PyObject *call_ctypes(Entry *e, PyObject *const *args, size_t nargsf, PyObject *kwnames) {
  return PyObject_Vectorcall(e->function, args, nargsf, kwnames);
}

template <typename... Args, size_t... I>
PyObject *call_entry(Entry *e, PyObject *const *args, size_t nargsf, PyObject *kwnames, int (*)(Args...), std::index_sequence<I...>) {
  std::tuple<Args...> values;
  if (PyVectorcall_NARGS(nargsf) != (Py_ssize_t)sizeof...(Args) || (kwnames && PyTuple_GET_SIZE(kwnames) > 0) ||
      !(from(args[I], std::get<I>(values)) && ...))
    return call_ctypes(e, args, nargsf, kwnames);
  int status = 0;
  const auto entry = reinterpret_cast<int (*)(Args...)>(e->address);
  Py_BEGIN_ALLOW_THREADS   // (as ctypes does: an entry point may wait for the GPU)
  status = entry(std::get<I>(values)...);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(status);
}

template <typename... Args>
std::index_sequence_for<Args...> positions(int (*)(Args...));

template <typename Pointer>
PyObject *vectorcall_of(PyObject *self, PyObject *const *args, size_t nargsf, PyObject *kwnames) {
  return call_entry(reinterpret_cast<Entry *>(self), args, nargsf, kwnames, Pointer(nullptr), decltype(positions(Pointer(nullptr)))());
}

// A type as ctypes codes it (pointers: c_void_p's letter).
template <typename T>
constexpr char code_of() {
  return std::is_pointer<T>::value ? 'P' : (std::is_same<T, double>::value ? 'd' : (std::is_same<T, int>::value ? 'i' : (std::is_same<T, int64_t>::value ? 'l' : 'L')));
}
template <typename... Args>
const char *codes_of(int (*)(Args...)) {
  static const char codes[] = {code_of<Args>()..., 0};
  return codes;
}

// The library is not linked: bind() brings the addresses, of whichever copy of it was loaded.
struct Known {
  const char *name, *codes;
  vectorcallfunc call;
} const kKnown[] = {
#define ENTRY(name) {#name, codes_of(decltype(&name)(nullptr)), vectorcall_of<decltype(&name)>}
    ENTRY(tfhip_fused_matmul),          ENTRY(tfhip_fused_matmul_noalloc),      ENTRY(tfhip_fused_conv2d),
    ENTRY(tfhip_fused_conv2d_add),      ENTRY(tfhip_fused_depthwise_conv2d),    ENTRY(tfhip_fused_pointwise_depthwise),
    ENTRY(tfhip_fused_conv2d_depthwise), ENTRY(tfhip_fused_inverted_residual), ENTRY(tfhip_mean_hw),
    ENTRY(tfhip_decode_weights),        ENTRY(tfhip_free),
#undef ENTRY
};

// What the callables here have of the function they stand for (all but the call itself): its attributes, its text, weak references.
template <typename Call>
PyObject *function_of(PyObject *self) { return reinterpret_cast<Call *>(self)->function; }
template <typename Call>
PyObject *text_of(PyObject *self) { return PyObject_Repr(function_of<Call>(self)); }

void entry_dealloc(PyObject *self) {
  PyObject_ClearWeakRefs(self);
  Py_XDECREF(function_of<Entry>(self));
  Py_TYPE(self)->tp_free(self);
}
PyObject *entry_getattro(PyObject *self, PyObject *name) {
  // (ctypes' way of taking an object as an argument: cast() and the like see the ctypes function)
  if (PyUnicode_CompareWithASCIIString(name, "_as_parameter_") == 0) {
    Py_INCREF(function_of<Entry>(self));
    return function_of<Entry>(self);
  }
  return PyObject_GetAttr(function_of<Entry>(self), name);
}
PyObject *entry_by_ctypes(PyObject *self, PyObject *const *args, size_t nargsf, PyObject *kwnames) {
  return call_ctypes(reinterpret_cast<Entry *>(self), args, nargsf, kwnames);
}
// (argtypes, restype, errcheck: the ctypes function goes by them, so from then on it is what is called)
int entry_setattro(PyObject *self, PyObject *name, PyObject *value) {
  reinterpret_cast<Entry *>(self)->call = entry_by_ctypes;
  return PyObject_SetAttr(function_of<Entry>(self), name, value);
}

PyTypeObject g_entry_type = {PyVarObject_HEAD_INIT(nullptr, 0)};

// (until the library is loaded every call of the two below goes to the function in Python, which loads it)
decltype(&tfhip_fused_matmul) g_fused_matmul = nullptr;
decltype(&tfhip_decode_weights) g_decode_weights = nullptr;
decltype(&tfhip_free) g_free = nullptr;

// bind(name, ctypes function, its address): the same function for callers that pass plain values.
PyObject *bind(PyObject *, PyObject *args) {
  const char *name = nullptr;
  PyObject *function = nullptr;
  unsigned long long address = 0;
  if (!PyArg_ParseTuple(args, "sOK", &name, &function, &address)) return nullptr;
  for (const Known &k : kKnown) {
    if (strcmp(k.name, name) != 0) continue;
    Entry *e = PyObject_New(Entry, &g_entry_type);
    if (!e) return nullptr;
    e->call = k.call;
    e->weak_references = nullptr;
    Py_INCREF(function);
    e->function = function;
    e->address = reinterpret_cast<void *>(static_cast<uintptr_t>(address));
    if (strcmp(name, "tfhip_fused_matmul") == 0) g_fused_matmul = reinterpret_cast<decltype(g_fused_matmul)>(e->address);
    if (strcmp(name, "tfhip_decode_weights") == 0) g_decode_weights = reinterpret_cast<decltype(g_decode_weights)>(e->address);
    if (strcmp(name, "tfhip_free") == 0) g_free = reinterpret_cast<decltype(g_free)>(e->address);
    return reinterpret_cast<PyObject *>(e);
  }
  return PyErr_Format(PyExc_KeyError, "%s", name);
}

// ---- pyhost.device_fused_matmul

enum { kA, kB, kOut, kBatchA, kBatchB, kM, kN, kK, kTransposeA, kTransposeB, kBias, kBiasStrides, kActivation, kPrelu, kPreluStrides, kAlpha, kParams };
const char *const kNames[kParams] = {"a", "b", "out", "batch_a", "batch_b", "m", "n", "k", "transpose_a", "transpose_b",
                                     "bias", "bias_strides", "activation", "prelu", "prelu_strides", "leakyrelu_alpha"};
PyObject *g_names[kParams] = {}, *g_ptr = nullptr;   // (interned)

// A function of the package by another body. Pickled and copied as a function is, by its name; as a class's attribute a method.
PyObject *by_name(PyObject *self, PyObject *);
PyMethodDef g_by_name[] = {{"__reduce__", by_name, METH_NOARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};
template <typename Call>
PyObject *python_getattro(PyObject *self, PyObject *name) {
  for (const char *own : {"__reduce__", "__reduce_ex__"})
    if (PyUnicode_CompareWithASCIIString(name, own) == 0) return PyObject_GenericGetAttr(self, name);
  return PyObject_GetAttr(function_of<Call>(self), name);
}
template <typename Call>
int python_setattro(PyObject *self, PyObject *name, PyObject *value) { return PyObject_SetAttr(function_of<Call>(self), name, value); }
PyObject *by_name(PyObject *self, PyObject *) { return PyObject_GetAttrString(self, "__qualname__"); }
PyObject *method_of(PyObject *self, PyObject *object, PyObject *) {
  if (object && object != Py_None) return PyMethod_New(self, object);
  Py_INCREF(self);
  return self;
}

struct MatmulCall {
  PyObject_HEAD
  vectorcallfunc call;
  PyObject *weak_references, *function, *activations, *check;   // the function in Python, the activations' numbers, what a status goes to
};

bool pointer_of(PyObject *operand, void *&to) {
  PyObject *ptr = PyObject_GetAttr(operand, g_ptr);
  if (!ptr) {
    PyErr_Clear();
    return false;
  }
  const bool ok = from_address(ptr, to);
  Py_DECREF(ptr);
  return ok;
}

bool strides_of(PyObject *o, int64_t (&to)[3]) {
  to[0] = to[1] = to[2] = 0;
  if (!o || o == Py_None) return true;
  const bool list = PyList_CheckExact(o);
  if ((!list && !PyTuple_CheckExact(o)) || PySequence_Fast_GET_SIZE(o) != 3) return false;
  for (int i = 0; i < 3; ++i)
    if (!from(PySequence_Fast_GET_ITEM(o, i), to[i])) return false;
  return true;
}

// The arguments by parameter; false: not in a form that is taken here.
bool arguments(PyObject *const *args, size_t nargsf, PyObject *kwnames, PyObject *(&to)[kParams]) {
  const Py_ssize_t n = PyVectorcall_NARGS(nargsf), named = kwnames ? PyTuple_GET_SIZE(kwnames) : 0;
  if (n > kParams) return false;
  for (Py_ssize_t i = 0; i < n; ++i) to[i] = args[i];
  for (Py_ssize_t i = 0; i < named; ++i) {
    PyObject *const name = PyTuple_GET_ITEM(kwnames, i);
    int p = 0;
    while (p < kParams && g_names[p] != name) ++p;
    if (p == kParams || to[p]) return false;   // (a name that is not interned, unknown or given twice)
    to[p] = args[n + i];
  }
  for (int p = kA; p <= kK; ++p)
    if (!to[p]) return false;
  return true;
}

PyObject *matmul_vectorcall(PyObject *self, PyObject *const *args, size_t nargsf, PyObject *kwnames) {
  MatmulCall *const f = reinterpret_cast<MatmulCall *>(self);
  PyObject *at[kParams] = {};
  void *a = nullptr, *b = nullptr, *out = nullptr, *bias = nullptr, *prelu = nullptr;
  int64_t size[5], bias_strides[3], prelu_strides[3];
  double alpha = 0.2;
  bool ok = g_fused_matmul && arguments(args, nargsf, kwnames, at) && pointer_of(at[kA], a) && pointer_of(at[kB], b) && pointer_of(at[kOut], out);
  for (int i = 0; i < 5 && ok; ++i) ok = from(at[kBatchA + i], size[i]);
  const auto given = [&](int p) { return at[p] && at[p] != Py_None; };
  ok = ok && (!given(kBias) || pointer_of(at[kBias], bias)) && (!given(kPrelu) || pointer_of(at[kPrelu], prelu)) &&
       strides_of(at[kBiasStrides], bias_strides) && strides_of(at[kPreluStrides], prelu_strides) &&
       (!at[kAlpha] || from(at[kAlpha], alpha));
  int transpose[2] = {0, 0}, activation = 0;
  for (int i = 0; i < 2 && ok; ++i) {
    PyObject *const t = at[kTransposeA + i];
    ok = !t || PyBool_Check(t);
    transpose[i] = t == Py_True;
  }
  if (ok && at[kActivation]) {
    PyObject *const number = PyUnicode_CheckExact(at[kActivation]) ? PyDict_GetItemWithError(f->activations, at[kActivation]) : nullptr;
    ok = number && from(number, activation);
    if (!ok) PyErr_Clear();
  }
  if (!ok) return PyObject_Vectorcall(f->function, args, nargsf, kwnames);
  int status = 0;
  Py_BEGIN_ALLOW_THREADS
  status = g_fused_matmul(static_cast<const float *>(a), static_cast<const float *>(b), static_cast<float *>(out), size[0], size[1], size[2], size[3],
                      size[4], transpose[0], transpose[1], static_cast<const float *>(bias), bias_strides, activation,
                      static_cast<const float *>(prelu), prelu_strides, alpha);
  Py_END_ALLOW_THREADS
  if (status) {
    PyObject *const raised = PyObject_CallFunction(f->check, "i", status);
    if (!raised) return nullptr;
    Py_DECREF(raised);
  }
  Py_RETURN_NONE;
}

void matmul_dealloc(PyObject *self) {
  MatmulCall *const f = reinterpret_cast<MatmulCall *>(self);
  PyObject_ClearWeakRefs(self);
  Py_XDECREF(f->function);
  Py_XDECREF(f->activations);
  Py_XDECREF(f->check);
  Py_TYPE(self)->tp_free(self);
}
PyTypeObject g_matmul_type = {PyVarObject_HEAD_INIT(nullptr, 0)};

// bind_matmul(function in Python, activations, check): the same function
PyObject *bind_matmul(PyObject *, PyObject *args) {
  PyObject *general = nullptr, *activations = nullptr, *check = nullptr;
  if (!PyArg_ParseTuple(args, "OO!O", &general, &PyDict_Type, &activations, &check)) return nullptr;
  MatmulCall *f = PyObject_New(MatmulCall, &g_matmul_type);
  if (!f) return nullptr;
  f->call = matmul_vectorcall;
  f->weak_references = nullptr;
  f->function = general;
  f->activations = activations;
  f->check = check;
  Py_INCREF(general);
  Py_INCREF(activations);
  Py_INCREF(check);
  return reinterpret_cast<PyObject *>(f);
}

// ---- pyhost.decode_weights_to_device

struct DecodeCall {
  PyObject_HEAD
  vectorcallfunc call;
  PyObject *weak_references, *function, *buffer_type, *check;   // the function in Python, DeviceBuffer, what a status goes to
};
PyObject *g_name, *g_dtype, *g_shape, *g_quantization, *g_scale, *g_min, *g_nbytes, *g_no_args;
constexpr int kNotInitialised = 1;   // (of the library's statuses: the general function sets it up)

bool is_text(PyObject *o, const char *text) { return PyUnicode_CheckExact(o) && PyUnicode_CompareWithASCIIString(o, text) == 0; }
bool number(PyObject *o, double &to) {
  int64_t whole = 0;
  if (from(o, to)) return true;
  if (!from(o, whole)) return false;
  to = (double)whole;   // (rounded as ctypes does)
  return true;
}

// An owned reference.
class Ref {
 public:
  explicit Ref(PyObject *o) : o_(o) {}
  Ref(Ref &&other) noexcept : o_(other.o_) { other.o_ = nullptr; }
  Ref(const Ref &) = delete;
  Ref &operator=(const Ref &) = delete;
  ~Ref() { Py_XDECREF(o_); }
  PyObject *get() const { return o_; }
  explicit operator bool() const { return o_ != nullptr; }

 private:
  PyObject *o_;
};

// (none, without an error, where there is none)
Ref entry_of(PyObject *dict, PyObject *key) {
  PyObject *const o = PyDict_GetItemWithError(dict, key);
  if (!o) PyErr_Clear();
  Py_XINCREF(o);
  return Ref(o);
}

// (all that the result is made of: other threads run during the call, and may change the manifest)
struct Weights {
  std::vector<Ref> names, shapes;   // (the lists are copies)
  std::vector<int64_t> offsets, elems;
  std::vector<int> kinds;
  std::vector<double> scale_min;
  size_t total = 0;
};

// What the manifest says, for tfhip_decode_weights; false: something for the general function to look at, or to refuse.
bool read_specs(PyObject *specs, Weights &w) {
  if (!PyList_CheckExact(specs)) return false;
  const Py_ssize_t count = PyList_GET_SIZE(specs);
  w.names.reserve(count);
  w.shapes.reserve(count);
  w.offsets.resize(count);
  w.elems.resize(count);
  w.kinds.resize(count);
  w.scale_min.resize(2 * count);
  for (Py_ssize_t i = 0; i < count; ++i) {
    if (i >= PyList_GET_SIZE(specs)) return false;   // (a key's own comparison has run)
    Py_INCREF(PyList_GET_ITEM(specs, i));
    const Ref spec(PyList_GET_ITEM(specs, i));
    if (!PyDict_CheckExact(spec.get())) return false;
    Ref name = entry_of(spec.get(), g_name);
    const Ref dtype = entry_of(spec.get(), g_dtype), extents = entry_of(spec.get(), g_shape), q = entry_of(spec.get(), g_quantization);
    if (!name || !PyUnicode_CheckExact(name.get()) || !dtype || !extents || !PyList_CheckExact(extents.get())) return false;
    Ref shape(PyList_GetSlice(extents.get(), 0, PyList_GET_SIZE(extents.get())));
    if (!shape) {
      PyErr_Clear();
      return false;
    }
    int64_t size = 1;
    for (Py_ssize_t d = 0; d < PyList_GET_SIZE(shape.get()); ++d) {
      int64_t extent = 0;
      if (!from(PyList_GET_ITEM(shape.get(), d), extent) || extent < 0 || (extent > 0 && size > (int64_t(1) << 40) / extent)) return false;
      size *= extent;
    }
    const bool to_float = is_text(dtype.get(), "float32"), to_int = is_text(dtype.get(), "int32");
    int kind = 0;
    size_t code = 4;
    if (!q || q.get() == Py_None) {
      if (!to_float && !to_int) {
        if (!is_text(dtype.get(), "bool")) return false;
        kind = 1;
        code = 1;
      }
    } else {
      if (!PyDict_CheckExact(q.get()) || (!to_float && !to_int)) return false;
      const Ref coded = entry_of(q.get(), g_dtype);
      if (!coded) return false;
      if (is_text(coded.get(), "float16")) {
        if (!to_float) return false;
        kind = 6;
        code = 2;
      } else {
        const bool bytes = is_text(coded.get(), "uint8");
        if (!bytes && !is_text(coded.get(), "uint16")) return false;
        kind = (bytes ? 2 : 4) + (to_int ? 1 : 0);
        code = bytes ? 1 : 2;
        const Ref scale = entry_of(q.get(), g_scale), min = entry_of(q.get(), g_min);
        if (!scale || !min || !number(scale.get(), w.scale_min[2 * i]) || !number(min.get(), w.scale_min[2 * i + 1])) return false;
      }
    }
    w.names.push_back(std::move(name));
    w.shapes.push_back(std::move(shape));
    w.offsets[i] = (int64_t)w.total;
    w.elems[i] = size;
    w.kinds[i] = kind;
    w.total += (size_t)size * code;
    if (w.total > (size_t(1) << 62)) return false;
  }
  return true;
}

// (DeviceBuffer.adopt(block, bytes), the shape), or nullptr with an error
PyObject *adopted(PyTypeObject *type, void *block, int64_t bytes, PyObject *shape) {
  PyObject *const buf = type->tp_new(type, g_no_args, nullptr);
  PyObject *const address = block ? PyLong_FromVoidPtr(block) : nullptr, *const ptr = block ? address : Py_None;
  PyObject *const nbytes = PyLong_FromLongLong(bytes);
  PyObject *pair = nullptr;
  if (buf && ptr && nbytes && PyObject_SetAttr(buf, g_nbytes, nbytes) == 0 && PyObject_SetAttr(buf, g_ptr, ptr) == 0)
    pair = PyTuple_Pack(2, buf, shape);
  Py_XDECREF(buf);
  Py_XDECREF(address);
  Py_XDECREF(nbytes);
  return pair;
}

PyObject *decode_vectorcall(PyObject *self, PyObject *const *args, size_t nargsf, PyObject *kwnames) {
  DecodeCall *const f = reinterpret_cast<DecodeCall *>(self);
  const auto general = [&] { return PyObject_Vectorcall(f->function, args, nargsf, kwnames); };
  if (!g_decode_weights || !g_free || PyVectorcall_NARGS(nargsf) != 2 || (kwnames && PyTuple_GET_SIZE(kwnames) > 0)) return general();
  try {
    Weights w;
    if (!read_specs(args[1], w) || w.elems.empty()) return general();
    std::vector<void *> outs(w.elems.size());
    Py_buffer host;
    if (PyObject_GetBuffer(args[0], &host, PyBUF_SIMPLE) != 0) {
      PyErr_Clear();
      return general();
    }
    int status = -1;
    if (host.len > 0 && w.total <= (size_t)host.len) {
      Py_BEGIN_ALLOW_THREADS
      status = g_decode_weights(host.buf, w.total, (int64_t)outs.size(), w.offsets.data(), w.elems.data(), w.kinds.data(), w.scale_min.data(), outs.data());
      Py_END_ALLOW_THREADS
    }
    PyBuffer_Release(&host);
    if (status == -1 || status == kNotInitialised) return general();
    if (status) return PyObject_CallFunction(f->check, "i", status);
    PyObject *result = PyDict_New();
    for (size_t i = 0; result && i < outs.size(); ++i) {
      PyObject *const pair = adopted(reinterpret_cast<PyTypeObject *>(f->buffer_type), outs[i], w.elems[i] * (w.kinds[i] == 1 ? 1 : 4), w.shapes[i].get());
      const bool kept = pair && PyDict_SetItem(result, w.names[i].get(), pair) == 0;
      Py_XDECREF(pair);
      if (!kept) Py_CLEAR(result);
    }
    if (!result)   // (what was wrapped is gone, and has given nothing back)
      for (void *block : outs)
        if (block) g_free(block);
    return result;
  } catch (const std::bad_alloc &) {
    return PyErr_NoMemory();
  }
}

void decode_dealloc(PyObject *self) {
  DecodeCall *const f = reinterpret_cast<DecodeCall *>(self);
  PyObject_ClearWeakRefs(self);
  Py_XDECREF(f->function);
  Py_XDECREF(f->buffer_type);
  Py_XDECREF(f->check);
  Py_TYPE(self)->tp_free(self);
}
PyTypeObject g_decode_type = {PyVarObject_HEAD_INIT(nullptr, 0)};

// bind_decode(function in Python, DeviceBuffer, check): the same function
PyObject *bind_decode(PyObject *, PyObject *args) {
  PyObject *general = nullptr, *buffer_type = nullptr, *check = nullptr;
  if (!PyArg_ParseTuple(args, "OO!O", &general, &PyType_Type, &buffer_type, &check)) return nullptr;
  DecodeCall *f = PyObject_New(DecodeCall, &g_decode_type);
  if (!f) return nullptr;
  f->call = decode_vectorcall;
  f->weak_references = nullptr;
  f->function = general;
  f->buffer_type = buffer_type;
  f->check = check;
  Py_INCREF(general);
  Py_INCREF(buffer_type);
  Py_INCREF(check);
  return reinterpret_cast<PyObject *>(f);
}

PyMethodDef g_methods[] = {{"bind", bind, METH_VARARGS, nullptr}, {"bind_matmul", bind_matmul, METH_VARARGS, nullptr},
                           {"bind_decode", bind_decode, METH_VARARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_pycall", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

template <typename Call>
bool ready(PyTypeObject &type, const char *name, destructor dealloc, getattrofunc get, setattrofunc set) {
  type.tp_name = name;
  type.tp_basicsize = sizeof(Call);
  type.tp_vectorcall_offset = offsetof(Call, call);
  type.tp_weaklistoffset = offsetof(Call, weak_references);
  type.tp_call = PyVectorcall_Call;
  type.tp_repr = text_of<Call>;
  type.tp_dealloc = dealloc;
  type.tp_getattro = get;
  type.tp_setattro = set;
  type.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL;
  return PyType_Ready(&type) == 0;
}
template <typename Call>
bool ready_as_function(PyTypeObject &type, const char *name, destructor dealloc) {
  type.tp_methods = g_by_name;
  type.tp_descr_get = method_of;
  return ready<Call>(type, name, dealloc, python_getattro<Call>, python_setattro<Call>);
}

}  // namespace

PyMODINIT_FUNC PyInit__pycall(void) {
  PyObject *const ctypes = PyImport_ImportModule("ctypes");
  if (!ctypes) return nullptr;
  g_array_type = PyObject_GetAttrString(ctypes, "Array");
  g_int64_type = PyObject_GetAttrString(ctypes, "c_int64");
  Py_DECREF(ctypes);
  g_underscore_type = PyUnicode_InternFromString("_type_");
  g_ptr = PyUnicode_InternFromString("ptr");
  if (!g_array_type || !g_int64_type || !g_underscore_type || !g_ptr) return nullptr;
  for (int i = 0; i < kParams; ++i)
    if (!(g_names[i] = PyUnicode_InternFromString(kNames[i]))) return nullptr;
  const std::pair<PyObject **, const char *> keys[] = {{&g_name, "name"}, {&g_dtype, "dtype"}, {&g_shape, "shape"}, {&g_quantization, "quantization"},
                                                       {&g_scale, "scale"}, {&g_min, "min"}, {&g_nbytes, "nbytes"}};
  for (const auto &key : keys)
    if (!(*key.first = PyUnicode_InternFromString(key.second))) return nullptr;
  if (!(g_no_args = PyTuple_New(0))) return nullptr;
  if (!ready<Entry>(g_entry_type, "tfjs_amd._pycall.Entry", entry_dealloc, entry_getattro, entry_setattro)) return nullptr;
  if (!ready_as_function<MatmulCall>(g_matmul_type, "tfjs_amd._pycall.MatmulCall", matmul_dealloc)) return nullptr;
  if (!ready_as_function<DecodeCall>(g_decode_type, "tfjs_amd._pycall.DecodeCall", decode_dealloc)) return nullptr;
  // NAMES: the entry points and their arguments as they were when this was compiled
  PyObject *const module = PyModule_Create(&g_module), *const names = PyDict_New();
  if (!module || !names) return nullptr;
  for (const Known &k : kKnown) {
    PyObject *const codes = PyUnicode_FromString(k.codes);
    if (!codes || PyDict_SetItemString(names, k.name, codes) != 0) return nullptr;
    Py_DECREF(codes);
  }
  return PyModule_AddObject(module, "NAMES", names) == 0 ? module : nullptr;
}
