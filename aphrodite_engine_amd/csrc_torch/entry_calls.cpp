// The C entry points as Python functions: a step of a mixer model is some seventy launches from Python, and ctypes looks at every argument of every one of
// them in Python's object model -- 20 to 45 arguments, 3 to 6 us a call where the launch itself takes 2.5.  Here the arguments are converted by the
// declared types of the function, at compile time.
// Measured on the host: 0.8 us against ctypes' 7.8 for the 40 arguments of the attention with a bias, 0.3 against 1.9 for 6 arguments.
//   bind(name, address, call, types) -> the function at that address under the type that the header declares for the name, or None for a name not listed
//                                       here, or listed with other types than the caller's (ctypes' letters, the result's first): headers that moved on
//                                       since this file was built leave such a name to ctypes
//   names() -> the names listed here
// The address comes from whoever loaded the library (_lib.py), so that nothing is linked and an overridden library path keeps its meaning; it is kept in
// the returned function, so that two libraries can be bound side by side.
// Whole numbers, None for a null pointer and numbers for floats are converted here, as ctypes converts them (whole numbers wrap); a call with anything
// else -- a ctypes object, another count -- is handed to `call`, ctypes' own function, as it is: what that takes, refuses or raises stays so.
// The interpreter lock is released around a call, as ctypes does.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstring>
#include <tuple>
#include <type_traits>
#include <utility>

#include "aphrodite_mi355x.h"
#include "aphrodite_mi355x_mixers.h"

namespace {

struct Target { void* at; PyObject* call; };      // a bound function's address, and ctypes' function for what is not converted here

// false: not a plain number (no exception is left)
template <typename T>
bool take(PyObject* o, T& out) {
  if constexpr (std::is_floating_point_v<T>) {
    if (!PyFloat_Check(o) && !PyLong_Check(o)) return false;
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) {          // a whole number beyond a double's range
      PyErr_Clear();
      return false;
    }
    out = (T)v;
    return true;
  } else {
    if (std::is_pointer_v<T> && o == Py_None) {
      out = T{};
      return true;
    }
    if (!PyLong_Check(o)) return false;
    const unsigned long long v = PyLong_AsUnsignedLongLongMask(o);
    if constexpr (std::is_pointer_v<T>) out = reinterpret_cast<T>((uintptr_t)v);
    else out = (T)v;
    return true;
  }
}

// ctypes' letter of a type
template <typename T>
constexpr char letter() {
  if constexpr (std::is_pointer_v<T>) return 'P';
  else if constexpr (std::is_floating_point_v<T>) return sizeof(T) == 4 ? 'f' : 'd';
  else if constexpr (sizeof(T) == 4) return std::is_signed_v<T> ? 'i' : 'I';
  else return sizeof(T) != 8 ? '?' : std::is_signed_v<T> ? 'l' : 'L';
}

template <typename F>
struct Entry;
template <typename R, typename... A>
struct Entry<R (*)(A...)> {
  static constexpr char types[] = {letter<R>(), letter<A>()..., 0};
  template <size_t... I>
  static PyObject* run(const Target* t, PyObject* const* args, std::index_sequence<I...>) {
    std::tuple<A...> a;
    if (!(take(args[I], std::get<I>(a)) && ...)) return PyObject_Vectorcall(t->call, args, sizeof...(A), nullptr);
    R r;
    Py_BEGIN_ALLOW_THREADS
    r = reinterpret_cast<R (*)(A...)>(t->at)(std::get<I>(a)...);
    Py_END_ALLOW_THREADS
    if constexpr (std::is_unsigned_v<R>) return PyLong_FromUnsignedLongLong(r);
    else return PyLong_FromLongLong(r);
  }
  static PyObject* call(PyObject* self, PyObject* const* args, Py_ssize_t n) {
    const Target* t = static_cast<const Target*>(PyCapsule_GetPointer(self, nullptr));
    if (!t) return nullptr;
    if (n != (Py_ssize_t)sizeof...(A)) return PyObject_Vectorcall(t->call, args, (size_t)n, nullptr);
    return run(t, args, std::index_sequence_for<A...>{});
  }
};

#define CORE_ENTRIES(X) \
  X(aphro_gptq_shuffle) X(aphro_gptq_repack) X(aphro_gptq_gemm) X(aphro_wna16_workspace_bytes) X(aphro_wna16_packed_a_bytes) X(aphro_wna16_pack_a) \
  X(aphro_wna16_ksplit) X(aphro_wna16_gemm_packed) X(aphro_wna16_gemm_silu_pack) X(aphro_paged_attention_packed) X(aphro_paged_attention_rope_packed) \
  X(aphro_fp8_gemm_ksplit) X(aphro_scaled_mm_fp8_slabs) X(aphro_scaled_mm_fp8_slabs_flags) X(aphro_fused_add_rms_norm_quant_fp8) \
  X(aphro_silu_and_mul_quant_fp8) X(aphro_fused_add_rms_norm_quant_fp8_static) X(aphro_silu_and_mul_quant_fp8_static) \
  X(aphro_paged_attention_rope_packed_scaled) X(aphro_paged_attention_rope_scaled_q8) X(aphro_paged_attention_rope_scaled_absmax) \
  X(aphro_sample_top_k_top_p) X(aphro_advance_step_flashattn) X(aphro_argmax_rows) X(aphro_topk_softmax) X(aphro_moe_align_block_size) \
  X(aphro_moe_gather_pack) X(aphro_wna16_grouped_ksplit) X(aphro_wna16_gemm_grouped) X(aphro_wna16_moe_tile_ksplit) X(aphro_wna16_moe_tile) \
  X(aphro_wna16_moe_tile_padded) X(aphro_moe_rows_to_f16) X(aphro_moe_route_align_blocks) X(aphro_moe_combine) X(aphro_fused_add_rms_norm_pack) \
  X(aphro_silu_and_mul_pack_slabs) X(aphro_silu_and_mul_pack) X(aphro_rotary_cache_supported) X(aphro_rotary_cache) X(aphro_rope_cache_scaled) \
  X(aphro_rope_cache) X(aphro_gptq_dequant) X(aphro_awq_dequantize) X(aphro_awq_gemm_workspace_bytes) X(aphro_awq_gemm) X(aphro_awq_repack) \
  X(aphro_awq_repack_zeros) X(aphro_reshape_and_cache) X(aphro_reshape_and_cache_flash) X(aphro_copy_blocks) X(aphro_swap_blocks) \
  X(aphro_wna16_gemm_large_workspace_bytes) X(aphro_wna16_rows_exact_tiles) X(aphro_wna16_gemm_large) X(aphro_wna16_gemm_large_silu_supported) \
  X(aphro_wna16_gemm_large_silu) X(aphro_wna16_gemm_mid_supported) X(aphro_wna16_gemm_mid_workspace_bytes) X(aphro_wna16_gemm_mid) \
  X(aphro_wna16_gemm_mid_ksplit) X(aphro_wna16_gemm_mid_packed) X(aphro_wna16_resident_ksplit) X(aphro_wna16_gemm_resident) \
  X(aphro_wna16_strip_relayout) X(aphro_wna16_strip_unrelayout) X(aphro_wna16_gemm_mid_packed_strip) X(aphro_wna16_gemm_large_strip_workspace_bytes) \
  X(aphro_wna16_gemm_large_strip) X(aphro_wna16_gemm_large_add_norm_supported) X(aphro_wna16_gemm_large_add_norm) \
  X(aphro_wna16_gemm_large_rotary_cache_supported) X(aphro_wna16_gemm_large_rotary_cache) X(aphro_wna16_gemm_rowmajor_supported) \
  X(aphro_fp8_gemm_rows_ksplit) X(aphro_fp8_gemm_rows_preferred) X(aphro_fp8_gemm_rows) X(aphro_dense_rows_preferred) X(aphro_dense_rows_slab_floats) \
  X(aphro_dense_rows) X(aphro_lm_head_argmax_supported) X(aphro_fp8_moe_gemm) X(aphro_moe_route_align) X(aphro_moe_route_gather_supported) \
  X(aphro_moe_route_gather) X(aphro_fused_add_rms_norm_router) X(aphro_fused_add_rms_norm_pack_combine) X(aphro_fp8_gemm_stream_ksplit) \
  X(aphro_fp8_gemm_stream) X(aphro_fp8_gemm_stream_silu_supported) X(aphro_fp8_gemm_resident_ksplit) X(aphro_fp8_strip_relayout) \
  X(aphro_fp8_gemm_resident) X(aphro_fp8_gemm_resident_strips) X(aphro_fp8_strip_relayout_interleaved) X(aphro_fp8_gemm_resident_aq) \
  X(aphro_fp8_gemm_resident_silu) X(aphro_fp8_quant_rows_aq) X(aphro_fp8_gemm_stream_silu_quant) X(aphro_gptq_dequant_bits) \
  X(aphro_gptq_gemm_bits_supported) X(aphro_gptq_gemm_bits) X(aphro_gptq_make_sequential_bits) X(aphro_lm_head_argmax) X(aphro_wna16_gemm_rowmajor) \
  X(aphro_convert_fp8) X(aphro_paged_attention_runs) X(aphro_paged_attention) X(aphro_static_scaled_fp8_quant) X(aphro_dynamic_scaled_fp8_quant) \
  X(aphro_dynamic_scaled_fp8_quant_ws) X(aphro_dynamic_per_token_scaled_fp8_quant) X(aphro_scaled_mm_fp8) \
  X(aphro_scaled_mm_fp8_large_workspace_bytes) X(aphro_fp8_w8a16_gemm_large_workspace_bytes) X(aphro_fp8_w8a16_gemm_large) \
  X(aphro_scaled_mm_fp8_large) X(aphro_fp8_w8a16_gemm) X(aphro_fp8_gemm_workspace_bytes) X(aphro_rms_norm) X(aphro_fused_add_rms_norm) \
  X(aphro_silu_and_mul) X(aphro_silu_and_mul_interleaved) X(aphro_rotary_embedding) X(aphro_flash_attn_varlen) X(aphro_flash_attn_varlen_window) \
  X(aphro_context_attention) X(aphro_context_attention_workspace_bytes) X(aphro_context_attention_gathered)
#define MIXER_ENTRIES(X) \
  X(aphro_embed_scale_f32) X(aphro_residual_layer_norm) X(aphro_act_and_mul) X(aphro_gated_group_rms_norm) X(aphro_paged_kv_write) \
  X(aphro_distance_bias_attention) X(aphro_residual_post_rms_norm) X(aphro_silu_gate_part_rms_norm) X(aphro_qk_row_norm_kv_write) \
  X(aphro_outer_memory_scan) X(aphro_outer_memory_chunked_workspace) X(aphro_outer_memory_chunked) X(aphro_depth_residual_rms_norm) \
  X(aphro_poly_norm) X(aphro_differential_norm_gate) X(aphro_short_conv) X(aphro_windowed_attention) X(aphro_differential_window_attention_supported) \
  X(aphro_differential_window_attention) X(aphro_experts_route) X(aphro_experts_align_capacity) X(aphro_experts_align) X(aphro_experts_block_rows) \
  X(aphro_experts_glu_gemm) X(aphro_experts_down_gemm) X(aphro_experts_combine) X(aphro_clamped_glu) X(aphro_residual_add2_rms_norm) \
  X(aphro_latent_prep) X(aphro_latent_attention_plain) X(aphro_latent_attention_fast_supported) X(aphro_latent_gather) \
  X(aphro_latent_attention_splits) X(aphro_latent_attention) X(aphro_sigmoid_gate_mul) X(aphro_experts_route_grouped) X(aphro_experts_route_topk) \
  X(aphro_logit_softcap) X(aphro_gated_delta_chunked_workspace) X(aphro_gated_delta_chunked) \
  X(aphro_gated_delta_scan) X(aphro_gated_head_rms_norm) X(aphro_conv_rotary_supported) X(aphro_conv_rotary_qk_norm_kv_write) \
  X(aphro_short_conv_state) X(aphro_residual_tanh_norm) X(aphro_rotary_qk_norm_kv_write)

struct Row { PyMethodDef def; const char* types; };
#define X(name) {{#name, (PyCFunction)(void (*)(void))&Entry<decltype(&name)>::call, METH_FASTCALL, nullptr}, Entry<decltype(&name)>::types},
Row rows[] = {CORE_ENTRIES(X) MIXER_ENTRIES(X)};
#undef X

void drop(PyObject* capsule) {
  Target* t = static_cast<Target*>(PyCapsule_GetPointer(capsule, nullptr));
  Py_XDECREF(t->call);
  delete t;
}

PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 4) return PyErr_Format(PyExc_TypeError, "bind(name, address, call, types)");
  const char *name = PyUnicode_AsUTF8(args[0]), *types = name ? PyUnicode_AsUTF8(args[3]) : nullptr;
  if (!types) return nullptr;
  void* at = PyLong_AsVoidPtr(args[1]);
  if (!at) return PyErr_Occurred() ? nullptr : PyErr_Format(PyExc_ValueError, "no address");
  for (Row& row : rows) {
    if (strcmp(row.def.ml_name, name)) continue;
    if (strcmp(row.types, types)) break;
    PyObject* self = PyCapsule_New(new Target{at, Py_NewRef(args[2])}, nullptr, &drop);
    if (!self) return nullptr;
    PyObject* call = PyCFunction_New(&row.def, self);
    Py_DECREF(self);
    return call;
  }
  Py_RETURN_NONE;
}

PyObject* names(PyObject*, PyObject*) {
  PyObject* list = PyList_New(0);
  for (const Row& row : rows) {
    PyObject* name = list ? PyUnicode_FromString(row.def.ml_name) : nullptr;
    if (!name || PyList_Append(list, name)) Py_CLEAR(list);
    Py_XDECREF(name);
  }
  return list;
}

PyMethodDef methods[] = {{"bind", (PyCFunction)(void (*)(void))&bind, METH_FASTCALL, nullptr}, {"names", &names, METH_NOARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "aphrodite_entry_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_aphrodite_entry_calls() { return PyModule_Create(&module); }
