// Python callables for the C-ABI entry points (include/spmla.h): _native.load(path) opens the library and returns
// {name: callable}. A call converts its arguments by the declared types (pointer: int or None; integer: int; float: float
// or int; anything else is a TypeError before the call), releases the GIL around the entry point and returns its value.
// ctypes needs 2.4 us for the 22 arguments of an attention call, near what the launch itself takes; this 0.2 us.
#include <Python.h>
#include <dlfcn.h>

#include <cstddef>
#include <tuple>
#include <type_traits>
#include <utility>

#include "spmla.h"

namespace {

bool bad(PyObject* o, const char* want) {
  PyErr_Format(PyExc_TypeError, "%s expected, got %s", want, Py_TYPE(o)->tp_name);
  return false;
}

template <class T>
bool convert(PyObject* o, T& v) {
  if constexpr (std::is_pointer_v<T>) {
    if (o == Py_None) { v = nullptr; return true; }
    if (!PyLong_Check(o)) return bad(o, "an address or None");
    v = reinterpret_cast<T>((uintptr_t)PyLong_AsUnsignedLongLongMask(o));
  } else if constexpr (std::is_floating_point_v<T>) {
    if (!PyFloat_Check(o) && !PyLong_Check(o)) return bad(o, "a number");
    const double d = PyFloat_AsDouble(o);
    if (d == -1.0 && PyErr_Occurred()) return false;
    v = (T)d;
  } else {
    if (!PyLong_Check(o)) return bad(o, "an integer");
    v = (T)PyLong_AsUnsignedLongLongMask(o);
  }
  return true;
}

template <class F>
struct Entry;
template <class R, class... A>
struct Entry<R (*)(A...)> {
  template <size_t... I>
  static PyObject* run(R (*f)(A...), PyObject* const* a, std::index_sequence<I...>) {
    std::tuple<A...> t{};
    if (!(convert(a[I], std::get<I>(t)) && ...)) return nullptr;
    R r;
    Py_BEGIN_ALLOW_THREADS
    r = std::apply(f, t);
    Py_END_ALLOW_THREADS
    return PyLong_FromLongLong((long long)r);
  }
  static PyObject* call(R (*f)(A...), PyObject* const* a, Py_ssize_t n) {
    if (n != (Py_ssize_t)sizeof...(A)) {
      PyErr_Format(PyExc_TypeError, "%zd arguments expected, got %zd", (Py_ssize_t)sizeof...(A), n);
      return nullptr;
    }
    return run(f, a, std::index_sequence_for<A...>());
  }
};

// One static slot per entry point: the symbol in the loaded library and the method definition.
#define SPMLA_CALLABLES(X)                                                                                          \
  X(spmla_cache_write) X(spmla_index_key_write) X(spmla_index_logits) X(spmla_topk) X(spmla_topk_ws_bytes)          \
  X(spmla_topk_ws) X(spmla_topk_ws_prehist) X(spmla_index_logits_hist) X(spmla_topk_scratch_bytes)                  \
  X(spmla_topk_scratch) X(spmla_topk_local) X(spmla_topk_merge) X(spmla_rows_from_topk) X(spmla_gather)             \
  X(spmla_gather_pcie) X(spmla_gather_tiers) X(spmla_copy_rows) X(spmla_row400_gather) X(spmla_row576_gather)       \
  X(spmla_row400_copy) X(spmla_row400_gather_tiers) X(spmla_row400_decode_tiers) X(spmla_tier_split)                \
  X(spmla_wcache_step) X(spmla_wcache_place) X(spmla_wcache_resolve) X(spmla_wcache_fill)                           \
  X(spmla_wcache_invalidate) X(spmla_split_res) X(spmla_wcache_split) X(spmla_compact_stage) X(spmla_attn_splitk)   \
  X(spmla_attn576) X(spmla_attn) X(spmla_attn576_ws) X(spmla_attn_paged) X(spmla_attn_ws_bytes) X(spmla_attn_merge) X(spmla_lse_merge)  \
  X(spmla_bmm_fp8) X(spmla_mla_query) X(spmla_topk_overlap) X(spmla_mtp_union) X(spmla_attn_packed)                 \
  X(spmla_index_key_write_shuffle) X(spmla_mqa_logits) X(spmla_paged_mqa_logits) X(spmla_paged_mqa_logits_seq)

#define SLOT(name)                                                                                                  \
  decltype(&::name) fn_##name = nullptr;                                                                            \
  PyObject* py_##name(PyObject*, PyObject* const* a, Py_ssize_t n) {                                                \
    return Entry<decltype(&::name)>::call(fn_##name, a, n);                                                         \
  }                                                                                                                 \
  PyMethodDef def_##name = {#name, (PyCFunction)(void (*)())py_##name, METH_FASTCALL, nullptr};
SPMLA_CALLABLES(SLOT)

bool add(PyObject* d, PyMethodDef* def) {
  PyObject* f = PyCFunction_New(def, nullptr);
  const bool ok = f && PyDict_SetItemString(d, def->ml_name, f) == 0;
  Py_XDECREF(f);
  return ok;
}

PyObject* load(PyObject*, PyObject* arg) {
  const char* path = PyUnicode_AsUTF8(arg);
  if (!path) return nullptr;
  void* h = dlopen(path, RTLD_NOW | RTLD_LOCAL);
  if (!h) return PyErr_Format(PyExc_OSError, "%s", dlerror());
  PyObject* d = PyDict_New();
  if (!d) return nullptr;
#define BIND(name)                                                                  \
  if (void* s = dlsym(h, #name)) {                                                  \
    fn_##name = (decltype(fn_##name))s;                                             \
    if (!add(d, &def_##name)) { Py_DECREF(d); return nullptr; }                     \
  }
  SPMLA_CALLABLES(BIND)
  return d;
}

PyMethodDef methods[] = {{"load", load, METH_O, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) { return PyModule_Create(&module); }
