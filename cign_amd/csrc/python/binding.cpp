// CPython binding of the C-ABI (include/cign_amd.h): one METH_FASTCALL
// function per entry point, its argument conversions generated from the
// declared prototype, so that a call costs the conversions of its arguments
// (about 0.1 us for an entry point of 30) and the kernel launches. ctypes took
// 3 us to convert such a call, beside 2 us a launch.
//
// Integers and pointers are Python ints (None: a null pointer), floats Python
// numbers; integers wrap to the parameter's width. The GIL is released around
// the call. The status or size comes back as an int.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stdint.h>

#include <tuple>
#include <type_traits>
#include <utility>

#include "cign_amd.h"

namespace {

template <typename T>
T convert(PyObject* o) {
  if constexpr (std::is_pointer_v<T>) {
    if (o == Py_None) return nullptr;
    if (!PyLong_Check(o)) {
      PyErr_Format(PyExc_TypeError, "expected an address (int) or None, got %s", Py_TYPE(o)->tp_name);
      return nullptr;
    }
    return reinterpret_cast<T>(PyLong_AsVoidPtr(o));
  } else if constexpr (std::is_floating_point_v<T>) {
    return static_cast<T>(PyFloat_AsDouble(o));
  } else {
    return static_cast<T>(PyLong_AsUnsignedLongLongMask(o));
  }
}

template <auto Fn, typename R, typename... A, size_t... I>
PyObject* invoke_impl(R (*)(A...), PyObject* const* args, Py_ssize_t n, std::index_sequence<I...>) {
  if (n != static_cast<Py_ssize_t>(sizeof...(A)))
    return PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", static_cast<Py_ssize_t>(sizeof...(A)), n);
  std::tuple<A...> v{convert<A>(args[I])...};
  if (PyErr_Occurred()) return nullptr;
  R rc;
  Py_BEGIN_ALLOW_THREADS;
  rc = Fn(std::get<I>(v)...);
  Py_END_ALLOW_THREADS;
  return PyLong_FromLongLong(static_cast<long long>(rc));
}

template <typename F>
struct Arity;
template <typename R, typename... A>
struct Arity<R (*)(A...)> : std::integral_constant<size_t, sizeof...(A)> {};

template <auto Fn>
PyObject* invoke(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return invoke_impl<Fn>(Fn, args, n, std::make_index_sequence<Arity<decltype(Fn)>::value>{});
}

#define CIGN_ENTRY(name) {#name, reinterpret_cast<PyCFunction>(invoke<&name>), METH_FASTCALL, nullptr}

PyMethodDef methods[] = {
    CIGN_ENTRY(cign_row_schedule_size),
    CIGN_ENTRY(cign_row_schedule_build),
    CIGN_ENTRY(cign_spmm_partial_bytes),
    CIGN_ENTRY(cign_spmm),
    CIGN_ENTRY(cign_spmm_fwd3),
    CIGN_ENTRY(cign_spmm_bwd3),
    CIGN_ENTRY(cign_spmm_fwd3_noalloc),
    CIGN_ENTRY(cign_gat_schedule_params),
    CIGN_ENTRY(cign_gat_fwd_workspace_bytes),
    CIGN_ENTRY(cign_gat_fwd),
    CIGN_ENTRY(cign_gat_row_agg_floats),
    CIGN_ENTRY(cign_gat_bwd_workspace_bytes),
    CIGN_ENTRY(cign_gat_bwd),
    CIGN_ENTRY(cign_gat_fwd_shard),
    CIGN_ENTRY(cign_gat_bwd_shard),
    CIGN_ENTRY(cign_gat_bwd_logits_ok),
    CIGN_ENTRY(cign_gat_bwd_logits),
    CIGN_ENTRY(cign_colsum_workspace_bytes),
    CIGN_ENTRY(cign_attn_logits_fwd),
    CIGN_ENTRY(cign_attn_logits_bwd),
    CIGN_ENTRY(cign_attn_logits_fwd_bf16),
    CIGN_ENTRY(cign_attn_logits_bwd_acc),
    CIGN_ENTRY(cign_attn_vec_grad),
    CIGN_ENTRY(cign_head_silu_fwd),
    CIGN_ENTRY(cign_head_silu_bwd),
    CIGN_ENTRY(cign_dropout_ln_fwd),
    CIGN_ENTRY(cign_dropout_ln_bwd),
    CIGN_ENTRY(cign_add_ln_fwd),
    CIGN_ENTRY(cign_add_ln_bwd),
    CIGN_ENTRY(cign_gamma_residual_fwd),
    CIGN_ENTRY(cign_gamma_residual_bwd),
    CIGN_ENTRY(cign_add_ln_cat_fwd),
    CIGN_ENTRY(cign_add_ln_cat_bwd),
    CIGN_ENTRY(cign_hop_gate_bwd_workspace_bytes),
    CIGN_ENTRY(cign_hop_gate_fwd),
    CIGN_ENTRY(cign_hop_gate_bwd),
    CIGN_ENTRY(cign_linear_fwd),
    CIGN_ENTRY(cign_linear_logits_fwd),
    CIGN_ENTRY(cign_linear_fwd_bf16y),
    CIGN_ENTRY(cign_linear_logits_fwd_bf16y),
    CIGN_ENTRY(cign_linear_gamma_fwd),
    CIGN_ENTRY(cign_linear_bwd_workspace_bytes),
    CIGN_ENTRY(cign_linear_bwd),
    CIGN_ENTRY(cign_linear_bwd_bf16gy),
    CIGN_ENTRY(cign_lin_logits_wgrad_workspace_bytes),
    CIGN_ENTRY(cign_lin_logits_wgrad),
    CIGN_ENTRY(cign_pack_proj_fwd_workspace_bytes),
    CIGN_ENTRY(cign_pack_proj_fwd),
    CIGN_ENTRY(cign_pack_proj_bwd_workspace_bytes),
    CIGN_ENTRY(cign_pack_proj_bwd),
    CIGN_ENTRY(cign_pack_gate_fwd),
    CIGN_ENTRY(cign_pack_gate_bwd),
    CIGN_ENTRY(cign_pack_fwd),
    CIGN_ENTRY(cign_pack_bwd),
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_cign", "Entry points of libcign_amd.", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__cign(void) { return PyModule_Create(&module); }
