// The entry points that a program enqueues on every step, called from Python without ctypes.  A launch occupies the device
// for 2 - 3 us and its host side takes about 2, so a row of small launches was bound by the conversions around them: a call
// that launches nothing took 1.8 us (quantize, 7 arguments), 5.2 (qmatmul, 14) or 5.8 (transpose, two arrays), here, where an
// argument is looked at once and in C, 0.6, 1.25 and 0.6.  Eager passes: QuantizeV2 -> MatMul -> Dequantize of
// 128 x 1024 x 1024 14.4 -> 12.2 us, three to six launches on small tensors 10.4 - 17.3 -> 7.5 - 13.3.
//
// Only the plain forms are converted here: None, int and objects with data_ptr() as addresses, int and float as numbers, the
// binding's own structures.  For anything else (numpy numbers, values that do not fit, wrong types) a call returns False
// without having done anything and the caller goes through its ctypes prototype, which converts or refuses as ever.
//
// The addresses of the entry points come from the library that the binding has loaded (init), so this module links to none.
// They belong to the module object, as do the check and the structures: a process may hold several copies of the binding
// (it has several import names, and ITEXHIP_LIB chooses a library for each), and each has a module object of its own.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <climits>
#include <tuple>
#include <type_traits>
#include <utility>

#include "itexhip.h"

namespace {

#define ENTRY_POINTS(X)                                                                                               \
  X(quantize) X(quantize_bf16) X(dequantize) X(dequantize16) X(requantize) X(requantize_per_channel)                  \
  X(minmax_i32_per_channel) X(minmax_f32) X(qgemm) X(qgemm_tile) X(qgemv) X(qgemm_sum) X(qmatmul) X(qmatmul_per_row)  \
  X(qmatmul_device_range) X(qmatmul_unpacked) X(quantize_dynamic) X(quantize_dynamic_static) X(quantize_dynamic_rows) \
  X(qbatch_matmul) X(pad_nhwc8) X(qconv2d) X(qconv2d_sum) X(qdepthwise_conv2d)

// All zero until init
struct State {
  PyObject* check;           // the binding's _check(status): raises unless it is 0
  PyObject* data_ptr;        // "data_ptr"
  PyTypeObject* structs[4];  // MatmulParams, Epilogue, BmmParams, ConvGeometry
#define POINTER(NAME) decltype(&itexhip_##NAME) NAME;
  ENTRY_POINTS(POINTER) POINTER(transpose)
#undef POINTER
};

State* state_of(PyObject* module) { return static_cast<State*>(PyModule_GetState(module)); }

// How many buffers of ctypes structures a call holds on to: at most two structures
struct Held {
  Py_buffer view[2];
  int n = 0;
  ~Held() { while (n > 0) PyBuffer_Release(&view[--n]); }
};

enum Result { kOk, kOther, kError };  // kOther: not a form for this path; kError: a Python exception is set

template <class T> constexpr int struct_index() {
  if (std::is_same_v<T, itexhip_matmul_params>) return 0;
  if (std::is_same_v<T, itexhip_epilogue>) return 1;
  if (std::is_same_v<T, itexhip_bmm_params>) return 2;
  if (std::is_same_v<T, itexhip_conv_geometry>) return 3;
  return -1;
}

Result address(const State& st, PyObject* o, void** out) {
  if (o == Py_None) { *out = nullptr; return kOk; }
  if (PyLong_CheckExact(o)) {
    *out = PyLong_AsVoidPtr(o);
    if (*out == nullptr && PyErr_Occurred()) { PyErr_Clear(); return kOther; }
    return kOk;
  }
  if (PyFloat_CheckExact(o) || PyUnicode_CheckExact(o)) return kOther;
  PyObject* r = PyObject_CallMethodNoArgs(o, st.data_ptr);
  if (r == nullptr) {
    if (!PyErr_ExceptionMatches(PyExc_AttributeError)) return kError;
    PyErr_Clear();
    return kOther;
  }
  const bool is_int = PyLong_CheckExact(r);
  *out = is_int ? PyLong_AsVoidPtr(r) : nullptr;
  Py_DECREF(r);
  if (!is_int) return kOther;
  if (*out == nullptr && PyErr_Occurred()) { PyErr_Clear(); return kOther; }
  return kOk;
}

template <class T>
Result convert(const State& st, PyObject* o, T* out, Held& held) {
  if constexpr (std::is_pointer_v<T>) {
    constexpr int s = struct_index<std::remove_cv_t<std::remove_pointer_t<T>>>();
    if constexpr (s >= 0) {
      if (Py_TYPE(o) != st.structs[s] || held.n == 2) return kOther;
      if (PyObject_GetBuffer(o, &held.view[held.n], PyBUF_SIMPLE) != 0) { PyErr_Clear(); return kOther; }
      const Py_buffer& v = held.view[held.n++];
      if (v.len < static_cast<Py_ssize_t>(sizeof(std::remove_pointer_t<T>))) return kOther;
      *out = static_cast<T>(v.buf);
      return kOk;
    } else {
      void* p;
      const Result r = address(st, o, &p);
      if (r == kOk) *out = static_cast<T>(p);
      return r;
    }
  } else if constexpr (std::is_floating_point_v<T>) {
    if (PyFloat_CheckExact(o)) { *out = static_cast<T>(PyFloat_AS_DOUBLE(o)); return kOk; }
    if (!PyLong_CheckExact(o)) return kOther;
    const double d = PyLong_AsDouble(o);
    if (d == -1.0 && PyErr_Occurred()) { PyErr_Clear(); return kOther; }
    *out = static_cast<T>(d);
    return kOk;
  } else {
    if (!PyLong_CheckExact(o)) return kOther;
    int overflow = 0;
    const long long v = PyLong_AsLongLongAndOverflow(o, &overflow);
    if (overflow != 0 || v != static_cast<long long>(static_cast<T>(v))) return kOther;
    *out = static_cast<T>(v);
    return kOk;
  }
}

PyObject* finish(const State& st, int status) {
  if (status == ITEXHIP_OK) Py_RETURN_TRUE;
  PyObject* r = PyObject_CallFunction(st.check, "i", status);
  Py_XDECREF(r);
  if (r == nullptr) return nullptr;
  Py_RETURN_TRUE;
}

// One METH_FASTCALL function per entry point; the C arguments' types are those of its declaration.
template <class F> struct Call;
template <class... A>
struct Call<int(A...)> {
  template <size_t... I>
  static PyObject* go(const State& st, int (*fn)(A...), PyObject* const* args, std::index_sequence<I...>) {
    std::tuple<std::remove_const_t<A>...> v{};
    Held held;
    Result r = kOk;
    (void)((r = convert(st, args[I], &std::get<I>(v), held), r == kOk) && ...);
    if (r == kError) return nullptr;
    if (r == kOther) Py_RETURN_FALSE;
    int status;
    Py_BEGIN_ALLOW_THREADS  // as ctypes does: a launch may wait for room in the queue
    status = fn(std::get<I>(v)...);
    Py_END_ALLOW_THREADS
    return finish(st, status);
  }
  static PyObject* run(const State& st, int (*fn)(A...), PyObject* const* args, Py_ssize_t n) {
    if (n != static_cast<Py_ssize_t>(sizeof...(A)) || fn == nullptr) Py_RETURN_FALSE;
    return go(st, fn, args, std::index_sequence_for<A...>{});
  }
};

#define DEFINE(NAME)                                                                              \
  PyObject* f_##NAME(PyObject* self, PyObject* const* args, Py_ssize_t n) {                       \
    const State& st = *state_of(self);                                                            \
    return Call<std::remove_pointer_t<decltype(&itexhip_##NAME)>>::run(st, st.NAME, args, n);     \
  }
ENTRY_POINTS(DEFINE)
#undef DEFINE

// transpose(x, y, elem_size, dims, perm, stream): the extents and the permutation as tuples of plain ints
constexpr Py_ssize_t kMaxRank = 8;
template <class T>
bool int_tuple(const State& st, PyObject* o, T (&out)[kMaxRank]) {
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(o); ++i) {
    Held none;
    if (convert(st, PyTuple_GET_ITEM(o, i), &out[i], none) != kOk) return false;
  }
  return true;
}
PyObject* f_transpose(PyObject* self, PyObject* const* args, Py_ssize_t n) {
  const State& st = *state_of(self);
  if (n != 6 || st.transpose == nullptr || !PyTuple_CheckExact(args[3]) || !PyTuple_CheckExact(args[4])) Py_RETURN_FALSE;
  const Py_ssize_t rank = PyTuple_GET_SIZE(args[3]);
  if (rank > kMaxRank || PyTuple_GET_SIZE(args[4]) != rank) Py_RETURN_FALSE;
  Held none;
  void *x, *y, *stream;
  int elem_size;
  int64_t dims[kMaxRank];
  int32_t perm[kMaxRank];
  const Result rx = address(st, args[0], &x);
  if (rx == kError) return nullptr;
  const Result ry = address(st, args[1], &y);
  if (ry == kError) return nullptr;
  const Result rs = address(st, args[5], &stream);
  if (rs == kError) return nullptr;
  if (rx != kOk || ry != kOk || rs != kOk || convert(st, args[2], &elem_size, none) != kOk ||
      !int_tuple(st, args[3], dims) || !int_tuple(st, args[4], perm))
    Py_RETURN_FALSE;
  int status;
  Py_BEGIN_ALLOW_THREADS
  status = st.transpose(x, y, elem_size, static_cast<int>(rank), dims, perm, stream);
  Py_END_ALLOW_THREADS
  return finish(st, status);
}

// init(address, check, structures): address(name) gives an entry point's address in the loaded library
PyObject* init(PyObject* self, PyObject* args) {
  State& st = *state_of(self);
  PyObject *addresses, *check, *s[4];
  if (!PyArg_ParseTuple(args, "OO(OOOO)", &addresses, &check, &s[0], &s[1], &s[2], &s[3])) return nullptr;
  for (PyObject* t : s)
    if (!PyType_Check(t)) { PyErr_SetString(PyExc_TypeError, "structures are types"); return nullptr; }
  bool ok = true;
  auto set = [&](const char* name, void** to) {
    PyObject* r = ok ? PyObject_CallFunction(addresses, "s", name) : nullptr;
    if (r != nullptr) *to = PyLong_AsVoidPtr(r);
    Py_XDECREF(r);
    if (PyErr_Occurred()) ok = false;
  };
#define SET(NAME) set("itexhip_" #NAME, reinterpret_cast<void**>(&st.NAME));
  ENTRY_POINTS(SET) SET(transpose)
#undef SET
  if (!ok) return nullptr;
  Py_INCREF(check);
  Py_XSETREF(st.check, check);
  for (int i = 0; i < 4; ++i) {
    Py_INCREF(s[i]);
    PyTypeObject* old = st.structs[i];
    st.structs[i] = reinterpret_cast<PyTypeObject*>(s[i]);
    Py_XDECREF(old);
  }
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
#define METHOD(NAME) {#NAME, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(f_##NAME)), METH_FASTCALL, nullptr},
    ENTRY_POINTS(METHOD) METHOD(transpose)
#undef METHOD
    {"init", init, METH_VARARGS, nullptr},
    {nullptr, nullptr, 0, nullptr}};

int exec_module(PyObject* module) {
  State& st = *state_of(module);
  st.data_ptr = PyUnicode_InternFromString("data_ptr");
  return st.data_ptr != nullptr ? 0 : -1;
}
int traverse(PyObject* module, visitproc visit, void* arg) {
  if (State* st = state_of(module)) {
    Py_VISIT(st->check);
    for (PyTypeObject* t : st->structs) Py_VISIT(t);
  }
  return 0;
}
int clear(PyObject* module) {
  if (State* st = state_of(module)) {
    Py_CLEAR(st->check);
    Py_CLEAR(st->data_ptr);
    for (PyTypeObject*& t : st->structs) Py_CLEAR(t);
  }
  return 0;
}
void free_module(void* module) { clear(static_cast<PyObject*>(module)); }

PyModuleDef_Slot slots[] = {{Py_mod_exec, reinterpret_cast<void*>(exec_module)}, {0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "itexhip_call", nullptr, sizeof(State), methods, slots, traverse, clear, free_module};

}  // namespace

PyMODINIT_FUNC PyInit_itexhip_call() { return PyModuleDef_Init(&module); }
