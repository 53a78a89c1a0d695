// The C entry points of libie_hip.so as CPython callables, for the calls a Python program
// makes per layer and step. A ctypes call of the fused decode step spends 5.7 us of host
// time in Python (argument conversion, one ie_kv_layout and a dozen data_ptr lookups), the
// same call here 1.9 us (matmul 1.9 and 0.8): with the launches' own 5 us, the difference
// between a host-bound and a GPU-bound decode step of one sequence (8-10 us).
//
// Arguments are the C function's, in order: a pointer is None or an object with data_ptr() (a
// tensor), a stream None or its handle, an integer a Python int; an ie_kv_layout is (tables,
// max_pages, pool, elements per token row); an ie_matrix the ctypes Matrix. The status code is
// returned. The GIL is released during the call, as ctypes does.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstring>
#include <tuple>
#include <type_traits>
#include <utility>

#include "ie_hip.h"

namespace {

// The torch dtypes of IE_KV_F32, IE_KV_F16, IE_KV_BF16, and the Matrix class (set_types).
PyObject* g_dtypes[3] = {nullptr, nullptr, nullptr};
PyObject* g_matrix = nullptr;
PyObject *g_data_ptr = nullptr, *g_numel = nullptr, *g_dtype = nullptr;

bool as_u64(PyObject* o, unsigned long long* v) {
  if (!PyLong_Check(o)) {
    PyErr_Format(PyExc_TypeError, "int expected instead of %s instance", Py_TYPE(o)->tp_name);
    return false;
  }
  *v = PyLong_AsUnsignedLongLongMask(o);
  return !(*v == ~0ull && PyErr_Occurred());
}

// elements // (IE_HIP_PAGE_SIZE * row), as Python divides: any row, rounded down.
bool pages_of(unsigned long long elements, PyObject* row, int32_t* pages) {
  if (!PyLong_Check(row)) {
    PyErr_Format(PyExc_TypeError, "int expected instead of %s instance", Py_TYPE(row)->tp_name);
    return false;
  }
  int over = 0;
  const long long r = PyLong_AsLongLongAndOverflow(row, &over), e = static_cast<long long>(elements);
  constexpr long long kMost = (1ll << 62) / IE_HIP_PAGE_SIZE;
  if (!over && r == 0) {
    PyErr_SetString(PyExc_ZeroDivisionError, "a token row has no elements");
    return false;
  }
  if (over > 0 || r > kMost) {
    *pages = 0;
  } else if (over < 0 || r < -kMost) {
    *pages = e ? -1 : 0;
  } else {
    const long long d = r * IE_HIP_PAGE_SIZE;
    *pages = int32_t(e / d - (d < 0 && e % d != 0));
  }
  return true;
}

bool address(PyObject* o, void** p) {
  *p = nullptr;
  if (o == Py_None) return true;
  unsigned long long v = 0;
  PyObject* r = PyObject_CallMethodNoArgs(o, g_data_ptr);
  if (!r) return false;
  const bool ok = as_u64(r, &v);
  Py_DECREF(r);
  if (!ok) return false;
  *p = reinterpret_cast<void*>(static_cast<uintptr_t>(v));
  return true;
}

template <class T>
bool convert(PyObject* o, T* out) {
  if constexpr (std::is_same_v<T, hipStream_t>) {
    unsigned long long v = 0;
    if (o != Py_None && !as_u64(o, &v)) return false;
    *out = reinterpret_cast<T>(static_cast<uintptr_t>(v));
    return true;
  } else if constexpr (std::is_pointer_v<T>) {
    void* p;
    if (!address(o, &p)) return false;
    *out = reinterpret_cast<T>(p);
    return true;
  } else if constexpr (std::is_floating_point_v<T>) {
    const double d = PyFloat_AsDouble(o);
    if (d == -1.0 && PyErr_Occurred()) return false;
    *out = static_cast<T>(d);
    return true;
  } else if constexpr (std::is_integral_v<T>) {
    unsigned long long v;
    if (!as_u64(o, &v)) return false;
    *out = static_cast<T>(v);
    return true;
  } else if constexpr (std::is_same_v<T, ie_matrix>) {
    const int is = PyObject_IsInstance(o, g_matrix);
    if (is <= 0) {
      if (!is) PyErr_SetString(PyExc_TypeError, "expected a Matrix");
      return false;
    }
    Py_buffer b;
    if (PyObject_GetBuffer(o, &b, PyBUF_SIMPLE)) return false;
    const bool ok = b.len == Py_ssize_t(sizeof(ie_matrix));
    if (ok) std::memcpy(out, b.buf, sizeof(ie_matrix));
    PyBuffer_Release(&b);
    if (!ok) PyErr_SetString(PyExc_TypeError, "expected a Matrix");
    return ok;
  } else {
    static_assert(std::is_same_v<T, ie_kv_layout>, "an argument type of ie_hip.h");
    if (!PyTuple_Check(o) || PyTuple_GET_SIZE(o) != 4) {
      PyErr_SetString(PyExc_TypeError, "expected (tables, max_pages, pool, row elements)");
      return false;
    }
    void* tables;
    unsigned long long max_pages, elements;
    PyObject* pool = PyTuple_GET_ITEM(o, 2);
    if (!address(PyTuple_GET_ITEM(o, 0), &tables) || !as_u64(PyTuple_GET_ITEM(o, 1), &max_pages))
      return false;
    PyObject* n = PyObject_CallMethodNoArgs(pool, g_numel);
    if (!n) return false;
    const bool ok = as_u64(n, &elements);
    Py_DECREF(n);
    PyObject* dtype = ok ? PyObject_GetAttr(pool, g_dtype) : nullptr;
    if (!dtype) return false;
    int code = -1;
    for (int i = 0; i < 3; ++i)
      if (dtype == g_dtypes[i]) code = i;
    if (code < 0) PyErr_SetObject(PyExc_KeyError, dtype);
    Py_DECREF(dtype);
    int32_t pages;
    if (code < 0 || !pages_of(elements, PyTuple_GET_ITEM(o, 3), &pages)) return false;
    *out = ie_kv_layout{static_cast<const int32_t*>(tables), int32_t(max_pages), IE_HIP_PAGE_SIZE,
                        int32_t(code), pages};
    return true;
  }
}

template <class F>
struct Args;
template <class R, class... A>
struct Args<R (*)(A...)> {
  using tuple = std::tuple<A...>;
  static constexpr size_t count = sizeof...(A);
};

template <bool kMatrices, class T>
bool convert_if(PyObject* o, T* out) {
  return std::is_same_v<T, ie_matrix> != kMatrices || convert(o, out);
}

// Matrices first: their check asks no tensor for anything.
template <class T, size_t... I>
bool convert_all(PyObject* const* args, T& t, std::index_sequence<I...>) {
  return (convert_if<true>(args[I], &std::get<I>(t)) && ...) &&
         (convert_if<false>(args[I], &std::get<I>(t)) && ...);
}

template <auto Fn>
PyObject* call(PyObject*, PyObject* const* args, Py_ssize_t n) {
  using A = Args<decltype(Fn)>;
  if (size_t(n) != A::count) {
    PyErr_Format(PyExc_TypeError, "expected %zu arguments, got %zd", A::count, n);
    return nullptr;
  }
  typename A::tuple t;
  if (!convert_all(args, t, std::make_index_sequence<A::count>{})) return nullptr;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = std::apply(Fn, t);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
}

PyObject* set_types(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 4) {
    PyErr_SetString(PyExc_TypeError, "expected the dtypes of f32, f16 and bf16 and the Matrix class");
    return nullptr;
  }
  Py_INCREF(args[3]);
  Py_XSETREF(g_matrix, args[3]);
  for (int i = 0; i < 3; ++i) {
    Py_INCREF(args[i]);
    Py_XSETREF(g_dtypes[i], args[i]);
  }
  Py_RETURN_NONE;
}

#define IE_CALL(name) \
  {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(&call<&name>)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    {"set_types", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(&set_types)), METH_FASTCALL,
     nullptr},
    IE_CALL(ie_hip_rope_and_cache),
    IE_CALL(ie_hip_attention),
    IE_CALL(ie_hip_attention_noalloc),
    IE_CALL(ie_hip_attention_planned),
    IE_CALL(ie_hip_rope_cache_attention),
    IE_CALL(ie_hip_rope_cache_attention_planned),
    IE_CALL(ie_hip_attention_prefill),
    IE_CALL(ie_hip_rope_cache_attention_prefill),
    IE_CALL(ie_hip_gather_rows),
    IE_CALL(ie_hip_gather_kv),
    IE_CALL(ie_hip_argmax_rows),
    IE_CALL(ie_hip_embedding),
    IE_CALL(ie_hip_rmsnorm),
    IE_CALL(ie_hip_matmul),
    IE_CALL(ie_hip_gate_up_silu),
    IE_CALL(ie_hip_qkv_proj),
    IE_CALL(ie_hip_rmsnorm_qkv_proj),
    IE_CALL(ie_hip_rmsnorm_gate_up_silu),
    {nullptr, nullptr, 0, nullptr}};
#undef IE_CALL

int exec(PyObject*) {
  if (!g_data_ptr) g_data_ptr = PyUnicode_InternFromString("data_ptr");
  if (!g_numel) g_numel = PyUnicode_InternFromString("numel");
  if (!g_dtype) g_dtype = PyUnicode_InternFromString("dtype");
  return g_data_ptr && g_numel && g_dtype ? 0 : -1;
}

PyModuleDef_Slot slots[] = {{Py_mod_exec, reinterpret_cast<void*>(&exec)}, {0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "native_calls", nullptr, 0, methods, slots,
                      nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_native_calls() { return PyModuleDef_Init(&module); }
