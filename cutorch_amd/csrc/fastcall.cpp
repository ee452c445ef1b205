// Calls of the C ABI from Python without ctypes' per-argument machinery: a Function object holds the entry
// point, its signature and the state pointer, converts its arguments, drops the interpreter lock around the call and asks
// for this thread's error message only while some thread holds one. A call on empty tensors (nothing is planned
// or launched) costs 0.77 us through ctypes and 0.13 here; back-to-back calls on small tensors are bound by the host.
// Conversions follow ctypes: whole numbers wrap to the parameter's width, a float is refused for one, numbers of any
// kind become floats; tensors come as addresses. Half parameters take a number and round it to the nearest half, as numpy does.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cmath>
#include <cstddef>
#include <cstdint>
#include <cstring>
#include <map>
#include <string>
#include <tuple>
#include <utility>

namespace {

struct Half {
  uint16_t bits;
};

const volatile long* g_pending = nullptr;   // threads that hold an error message
const char* (*g_last_error)() = nullptr;
void (*g_clear_error)() = nullptr;
PyObject* g_error = nullptr;

// The half nearest to x, ties to even (what numpy's conversion from float64 gives).
uint16_t half_bits(double x) {
  uint64_t b;
  std::memcpy(&b, &x, 8);
  const uint16_t sign = (uint16_t)((b >> 48) & 0x8000);
  if (std::isnan(x)) return (uint16_t)(sign | 0x7c00 | ((b >> 42) & 0x3ff) | ((b >> 42) & 0x3ff ? 0 : 1));
  const double a = std::fabs(x);
  if (a >= 65520.0) return (uint16_t)(sign | 0x7c00);
  if (a < 6.103515625e-05) return (uint16_t)(sign | (uint16_t)std::nearbyint(a * 16777216.0));   // steps of 2^-24 (1024 = the smallest normal)
  int e;
  const double m = std::frexp(a, &e);                               // a = m 2^e, 1/2 <= m < 1
  const int q = (int)std::nearbyint(m * 2048.0);                    // 11 bits; 2048 carries into the exponent
  return (uint16_t)(sign | (((e + 14) << 10) + (q - 1024)));
}

template <typename T>
struct From;      // get(object, value): false with a Python error set
template <typename T>
struct FromInt {
  static bool get(PyObject* o, T& v) {
    if (PyFloat_Check(o)) {
      PyErr_Format(PyExc_TypeError, "int expected instead of %s instance", Py_TYPE(o)->tp_name);
      return false;
    }
    const unsigned long long u = PyLong_AsUnsignedLongLongMask(o);
    if (u == (unsigned long long)-1 && PyErr_Occurred()) return false;
    v = (T)u;
    return true;
  }
};
template <> struct From<long> : FromInt<long> {};
template <> struct From<int> : FromInt<int> {};
template <> struct From<short> : FromInt<short> {};
template <> struct From<signed char> : FromInt<signed char> {};
template <> struct From<unsigned char> : FromInt<unsigned char> {};
template <>
struct From<double> {
  static bool get(PyObject* o, double& v) {
    v = PyFloat_AsDouble(o);
    return !(v == -1.0 && PyErr_Occurred());
  }
};
template <>
struct From<float> {
  static bool get(PyObject* o, float& v) {
    double d;
    if (!From<double>::get(o, d)) return false;
    v = (float)d;
    return true;
  }
};
template <>
struct From<Half> {
  static bool get(PyObject* o, Half& v) {
    double d;
    if (!From<double>::get(o, d)) return false;
    v.bits = half_bits(d);
    return true;
  }
};
template <>
struct From<void*> {
  static bool get(PyObject* o, void*& v) {
    v = PyLong_AsVoidPtr(o);
    return v || !PyErr_Occurred();
  }
};
// what the entry point takes: a half travels as its bits
template <typename T> struct Wire { using type = T; static T of(T v) { return v; } };
template <> struct Wire<Half> { using type = uint16_t; static uint16_t of(Half v) { return v.bits; } };

PyObject* to_python(float v) { return PyFloat_FromDouble(v); }
PyObject* to_python(double v) { return PyFloat_FromDouble(v); }
PyObject* to_python(long v) { return PyLong_FromLong(v); }
PyObject* to_python(int v) { return PyLong_FromLong(v); }
PyObject* to_python(short v) { return PyLong_FromLong(v); }
PyObject* to_python(signed char v) { return PyLong_FromLong(v); }
PyObject* to_python(unsigned char v) { return PyLong_FromLong(v); }
PyObject* to_python(uint16_t v) { return PyLong_FromLong(v); }

// true: this thread has a message, now raised
bool failed() {
  if (!*g_pending) return false;
  const char* msg = g_last_error();
  if (!msg) return false;
  PyErr_SetString(g_error, msg);
  g_clear_error();
  return true;
}

using Invoker = PyObject* (*)(void* fn, void* state, PyObject* const* args);

template <typename R, typename... A>
struct Call {
  template <size_t... I>
  static PyObject* go(void* fn, void* state, PyObject* const* args, std::index_sequence<I...>) {
    std::tuple<A...> v;
    if (!(From<A>::get(args[I], std::get<I>(v)) && ...)) return nullptr;
    using Fn = R (*)(void*, typename Wire<A>::type...);
    if constexpr (std::is_void<R>::value) {
      Py_BEGIN_ALLOW_THREADS
      reinterpret_cast<Fn>(fn)(state, Wire<A>::of(std::get<I>(v))...);
      Py_END_ALLOW_THREADS
      if (failed()) return nullptr;
      Py_RETURN_NONE;
    } else {
      R r;
      Py_BEGIN_ALLOW_THREADS
      r = reinterpret_cast<Fn>(fn)(state, Wire<A>::of(std::get<I>(v))...);
      Py_END_ALLOW_THREADS
      if (failed()) return nullptr;
      return to_python(r);
    }
  }
  static PyObject* invoke(void* fn, void* state, PyObject* const* args) {
    return go(fn, state, args, std::index_sequence_for<A...>{});
  }
};

std::map<std::string, std::pair<Invoker, int>>& registry() {
  static std::map<std::string, std::pair<Invoker, int>> r;
  return r;
}
template <typename R, typename... A>
void add(const std::string& sig) {
  registry()[sig] = {&Call<R, A...>::invoke, (int)sizeof...(A)};
}
// Signatures: the return type, then the parameters after the state. t tensor, v nothing, f float, d double, l long, i int,
// h short, b signed char, B unsigned char, e half. `c`, X: the element type of the entry point's scalars.
template <typename X>
void add_element(const std::string& c) {
  using T = void*;
  add<void, T, X>("vt" + c);
  add<void, T, X, T>("vt" + c + "t");
  add<void, T, T, X>("vtt" + c);
  add<void, T, T, X, X>("vtt" + c + c);
  add<void, T, T, X, T>("vtt" + c + "t");
  add<void, T, T, X, T, T>("vtt" + c + "tt");
  add<void, T, T, T, X>("vttt" + c);
  add<void, T, T, X, long, int>("vtt" + c + "li");
  add<void, T, T, X, long, X>("vtt" + c + "l" + c);
}
template <typename R>
void add_result(const std::string& r) {
  using T = void*;
  add<R, T>(r + "t");
  add<R, T, int>(r + "ti");
}
void fill_registry() {
  using T = void*;
  add<void, T>("vt");
  add<void, T, T>("vtt");
  add<void, T, T, T>("vttt");
  add<void, T, T, long>("vttl");
  add<void, T, T, long, int>("vttli");
  add<void, T, T, long, int, int>("vttlii");
  add<void, T, T, T, long, int>("vtttli");
  add<int, T, T>("itt");
  add_element<float>("f");
  add_element<double>("d");
  add_element<long>("l");
  add_element<int>("i");
  add_element<short>("h");
  add_element<signed char>("b");
  add_element<unsigned char>("B");
  add_element<Half>("e");
  add_result<float>("f");
  add_result<double>("d");
  add_result<long>("l");
  add_result<int>("i");
  add_result<short>("h");
  add_result<signed char>("b");
  add_result<unsigned char>("B");
  add_result<uint16_t>("e");
  add<float, T, float>("ftf");
  add<float, T, Half>("fte");
  add<double, T, double>("dtd");
  add<float, T, T, float>("fttf");
  add<float, T, T, Half>("ftte");
  add<double, T, T, double>("dttd");
}

struct Function {
  PyObject_HEAD
  vectorcallfunc call;
  Invoker invoke;
  void* fn;
  void* state;
  int nargs;
};

PyObject* function_call(PyObject* self, PyObject* const* args, size_t nargsf, PyObject* kwnames) {
  const Function* f = reinterpret_cast<const Function*>(self);
  const Py_ssize_t n = PyVectorcall_NARGS(nargsf);
  if (n != f->nargs || (kwnames && PyTuple_GET_SIZE(kwnames) != 0)) {
    PyErr_Format(PyExc_TypeError, "this function takes %d arguments (%zd given)", f->nargs, n);
    return nullptr;
  }
  return f->invoke(f->fn, f->state, args);
}

PyTypeObject FunctionType = {PyVarObject_HEAD_INIT(nullptr, 0)};

PyObject* setup(PyObject*, PyObject* args) {
  PyObject *pending, *last, *clear, *error;
  if (!PyArg_ParseTuple(args, "OOOO", &pending, &last, &clear, &error)) return nullptr;
  g_pending = static_cast<const volatile long*>(PyLong_AsVoidPtr(pending));
  g_last_error = reinterpret_cast<const char* (*)()>(PyLong_AsVoidPtr(last));
  g_clear_error = reinterpret_cast<void (*)()>(PyLong_AsVoidPtr(clear));
  if (PyErr_Occurred()) return nullptr;
  Py_INCREF(error);
  Py_XDECREF(g_error);
  g_error = error;
  Py_RETURN_NONE;
}

// bind(address, signature, state): a Function, or None for a signature that is not served
PyObject* bind(PyObject*, PyObject* args) {
  PyObject *address, *state;
  const char* sig;
  if (!PyArg_ParseTuple(args, "OsO", &address, &sig, &state)) return nullptr;
  const auto it = registry().find(sig);
  if (it == registry().end() || !g_error) Py_RETURN_NONE;
  Function* f = PyObject_New(Function, &FunctionType);
  if (!f) return nullptr;
  f->call = function_call;
  f->invoke = it->second.first;
  f->nargs = it->second.second;
  f->fn = PyLong_AsVoidPtr(address);
  f->state = PyLong_AsVoidPtr(state);
  if (PyErr_Occurred()) {
    Py_DECREF(f);
    return nullptr;
  }
  return reinterpret_cast<PyObject*>(f);
}

PyObject* py_half_bits(PyObject*, PyObject* o) {
  Half h;
  if (!From<Half>::get(o, h)) return nullptr;
  return PyLong_FromLong(h.bits);
}

PyMethodDef kMethods[] = {{"setup", setup, METH_VARARGS, nullptr},
                          {"bind", bind, METH_VARARGS, nullptr},
                          {"half_bits", py_half_bits, METH_O, nullptr},
                          {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_fastcall", "Calls of libTHC.so's entry points.", -1, kMethods};

}  // namespace

PyMODINIT_FUNC PyInit__fastcall() {
  fill_registry();
  FunctionType.tp_name = "cutorch_amd._fastcall.Function";
  FunctionType.tp_basicsize = sizeof(Function);
  FunctionType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL;
  FunctionType.tp_vectorcall_offset = offsetof(Function, call);
  FunctionType.tp_call = PyVectorcall_Call;
  if (PyType_Ready(&FunctionType) < 0) return nullptr;
  return PyModule_Create(&kModule);
}
