// Python entry to the C ABI without ctypes: bind(name, address) returns a
// callable that converts its arguments by the declared C signature
// (llamazero_hip.h) and calls the function at `address`.  A ctypes call of
// these 15-30 argument functions spends 3 us converting arguments, more than
// the kernel launch behind it; here the conversion is compiled per signature.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstring>
#include <tuple>
#include <type_traits>
#include <utility>

#include "../../include/llamazero_hip.h"

namespace {

// One argument, with ctypes' leniencies: None is a null pointer, an integer
// is taken modulo its width, an int passes for a float.
template <typename T>
bool convert(PyObject* o, T& out) {
  if constexpr (std::is_pointer_v<T>) {
    if (o == Py_None) {
      out = nullptr;
      return true;
    }
    out = reinterpret_cast<T>(PyLong_AsVoidPtr(o));
    return out != nullptr || !PyErr_Occurred();
  } else if constexpr (std::is_floating_point_v<T>) {
    const double d = PyFloat_AsDouble(o);
    out = static_cast<T>(d);
    return d != -1.0 || !PyErr_Occurred();
  } else {
    const unsigned long long v = PyLong_AsUnsignedLongLongMask(o);
    out = static_cast<T>(v);
    return v != static_cast<unsigned long long>(-1) || !PyErr_Occurred();
  }
}

template <typename Sig, int Id>
struct Entry;

template <typename R, typename... A, int Id>
struct Entry<R(A...), Id> {
  static inline R (*fn)(A...) = nullptr;

  template <size_t... I>
  static PyObject* invoke(PyObject* const* args, std::index_sequence<I...>) {
    std::tuple<A...> v;
    if (!(convert(args[I], std::get<I>(v)) && ...)) return nullptr;
    R r;
    Py_BEGIN_ALLOW_THREADS
    r = fn(std::get<I>(v)...);
    Py_END_ALLOW_THREADS
    return PyLong_FromLongLong(static_cast<long long>(r));
  }
  static PyObject* call(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != static_cast<Py_ssize_t>(sizeof...(A)))
      return PyErr_Format(PyExc_TypeError, "this function takes %zd arguments (%zd given)",
                          static_cast<Py_ssize_t>(sizeof...(A)), n);
    return invoke(args, std::index_sequence_for<A...>{});
  }
  static void set(void* p) { fn = reinterpret_cast<R (*)(A...)>(p); }
};

struct Slot {
  PyMethodDef def;
  void (*set)(void*);
};

#define LZ_ENTRY(name)                                                                                     \
  {{#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&Entry<decltype(name), __LINE__>::call)), \
    METH_FASTCALL, nullptr},                                                                               \
   &Entry<decltype(name), __LINE__>::set}

Slot kSlots[] = {
    LZ_ENTRY(lz_version),
    LZ_ENTRY(lz_device_cus),
    LZ_ENTRY(lz_adamw),
    LZ_ENTRY(lz_adamw_step),
    LZ_ENTRY(lz_adamw_dev),
    LZ_ENTRY(lz_sumsq),
    LZ_ENTRY(lz_adamw_norm_workspace),
    LZ_ENTRY(lz_adamw_norm),
    LZ_ENTRY(lz_adamw_multi),
    LZ_ENTRY(lz_sumsq_multi),
    LZ_ENTRY(lz_clip_finalize),
    LZ_ENTRY(lz_mt_gather),
    LZ_ENTRY(lz_mt_scatter),
    LZ_ENTRY(lz_mt_gather_host),
    LZ_ENTRY(lz_mt_scatter_host),
    LZ_ENTRY(lz_axpy_f32),
    LZ_ENTRY(lz_add_inplace),
    LZ_ENTRY(lz_scale_inplace),
    LZ_ENTRY(lz_scale_dev),
    LZ_ENTRY(lz_fill),
    LZ_ENTRY(lz_cast),
    LZ_ENTRY(lz_rmsnorm_fwd),
    LZ_ENTRY(lz_rmsnorm_bwd_workspace),
    LZ_ENTRY(lz_rmsnorm_bwd),
    LZ_ENTRY(lz_rmsnorm_bwd_noalloc),
    LZ_ENTRY(lz_rope_table),
    LZ_ENTRY(lz_rope),
    LZ_ENTRY(lz_swiglu_fwd),
    LZ_ENTRY(lz_swiglu_bwd),
    LZ_ENTRY(lz_embedding_fwd),
    LZ_ENTRY(lz_embedding_bwd),
    LZ_ENTRY(lz_ce_fwd),
    LZ_ENTRY(lz_ce_reduce),
    LZ_ENTRY(lz_ce_bwd),
    LZ_ENTRY(lz_transpose),
    LZ_ENTRY(lz_copy2d),
    LZ_ENTRY(lz_gemm_nt),
    LZ_ENTRY(lz_gemm_swiglu),
    LZ_ENTRY(lz_gemm_rope),
    LZ_ENTRY(lz_gemm_rope_hd),
    LZ_ENTRY(lz_gemm_swiglu_bwd),
    LZ_ENTRY(lz_gemm),
    LZ_ENTRY(lz_gemm_f32),
    LZ_ENTRY(lz_gemm_f32_workspace),
    LZ_ENTRY(lz_gemm_f32_plan),
    LZ_ENTRY(lz_gemm_workspace),
    LZ_ENTRY(lz_gemm_plan),
    LZ_ENTRY(lz_attn_path),
    LZ_ENTRY(lz_attn_tiles),
    LZ_ENTRY(lz_attn_fwd),
    LZ_ENTRY(lz_attn_delta),
    LZ_ENTRY(lz_attn_fwd_general),
    LZ_ENTRY(lz_attn_bwd_general),
    LZ_ENTRY(lz_attn_bwd_with_o),
    LZ_ENTRY(lz_attn_direct),
    LZ_ENTRY(lz_attn_fwd_direct),
    LZ_ENTRY(lz_attn_bwd_direct),
    LZ_ENTRY(lz_dropout),
    LZ_ENTRY(lz_dropout_mask),
    LZ_ENTRY(lz_attn_bwd),
};

PyObject* bind(PyObject*, PyObject* args) {
  const char* name;
  PyObject* address;
  if (!PyArg_ParseTuple(args, "sO", &name, &address)) return nullptr;
  void* p = PyLong_AsVoidPtr(address);
  if (p == nullptr) {
    if (!PyErr_Occurred()) PyErr_Format(PyExc_ValueError, "null address for %s", name);
    return nullptr;
  }
  for (Slot& s : kSlots)
    if (std::strcmp(s.def.ml_name, name) == 0) {
      s.set(p);
      return PyCFunction_New(&s.def, nullptr);
    }
  return PyErr_Format(PyExc_KeyError, "no entry point %s", name);
}

PyMethodDef kMethods[] = {{"bind", bind, METH_VARARGS, "bind(name, address) -> callable"}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_pycall", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__pycall(void) { return PyModule_Create(&kModule); }
