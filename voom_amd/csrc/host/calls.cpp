// Calls of the C ABI from Python, one wrapper per entry point, generated from the
// declarations in voom_hip.h.  A small op is bound by the host: through ctypes a
// call with 20 arguments took 4.4 us, of which the launch is about 1.5, and the
// tensor checks in front of it 2.5 us more.  A decode call on one short sequence:
// 13.6 -> 11.0 us; a 512-token prompt through 30 layers (152 calls): 2.36 -> 2.07 ms.
// Pointers come as tensors (their data), integers or None; integers are cut to the
// parameter's width, as ctypes does.  The interpreter lock is released during each
// call.
#include <Python.h>

#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>
#include <exception>
#include <optional>
#include <tuple>
#include <type_traits>
#include <utility>

#include "../../../include/voom_hip.h"

namespace {

// A plain tensor or parameter, whose attributes can be read without Python;
// subclasses go through their own attributes.
bool plain_tensor(PyObject* o) { return THPVariable_CheckExact(o); }

bool to_integer(PyObject* o, unsigned long long& out) {
  if (PyFloat_Check(o)) {
    PyErr_SetString(PyExc_TypeError, "int expected instead of float");
    return false;
  }
  out = PyLong_AsUnsignedLongLongMask(o);
  return !(out == static_cast<unsigned long long>(-1) && PyErr_Occurred());
}

bool to_pointer(PyObject* o, void*& out) {
  if (o == Py_None) {
    out = nullptr;
    return true;
  }
  if (plain_tensor(o)) {
    out = const_cast<void*>(THPVariable_Unpack(o).data_ptr());
    return true;
  }
  unsigned long long v = 0;
  if (PyLong_Check(o)) {
    if (!to_integer(o, v)) return false;
  } else if (THPVariable_Check(o)) {
    PyObject* p = PyObject_CallMethod(o, "data_ptr", nullptr);
    if (!p) return false;
    const bool ok = to_integer(p, v);
    Py_DECREF(p);
    if (!ok) return false;
  } else {
    PyErr_SetString(PyExc_TypeError, "a pointer is a tensor, an integer or None");
    return false;
  }
  out = reinterpret_cast<void*>(static_cast<uintptr_t>(v));
  return true;
}

template <class T>
bool convert(PyObject* o, T& out) {
  if constexpr (std::is_pointer_v<T>) {
    void* p = nullptr;
    if (!to_pointer(o, p)) return false;
    out = static_cast<T>(p);
  } else if constexpr (std::is_floating_point_v<T>) {
    const double d = PyFloat_AsDouble(o);
    if (d == -1.0 && PyErr_Occurred()) return false;
    out = static_cast<T>(d);
  } else {
    unsigned long long v = 0;
    if (!to_integer(o, v)) return false;
    out = static_cast<T>(v);
  }
  return true;
}

template <class R, class... A, size_t... I>
PyObject* invoke(R (*fn)(A...), PyObject* const* args, Py_ssize_t n, std::index_sequence<I...>) {
  if (n != static_cast<Py_ssize_t>(sizeof...(A))) {
    PyErr_Format(PyExc_TypeError, "%zu arguments expected, got %zd", sizeof...(A), n);
    return nullptr;
  }
  // const void* parameters are filled through void*
  std::tuple<std::conditional_t<std::is_pointer_v<A>,
                                std::add_pointer_t<std::remove_const_t<std::remove_pointer_t<A>>>, A>...> v;
  if (!(convert(args[I], std::get<I>(v)) && ...)) return nullptr;
  R r;
  Py_BEGIN_ALLOW_THREADS;
  r = fn(std::get<I>(v)...);
  Py_END_ALLOW_THREADS;
  if constexpr (std::is_signed_v<R>) return PyLong_FromLongLong(r);
  else return PyLong_FromUnsignedLongLong(r);
}

template <class R, class... A>
PyObject* dispatch(R (*fn)(A...), PyObject* const* args, Py_ssize_t n) {
  try {
    return invoke(fn, args, n, std::index_sequence_for<A...>{});
  } catch (const std::exception& e) {  // a tensor without storage
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
}

template <auto FN>
PyObject* wrap(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return dispatch(FN, args, n);
}

// The device of the given tensors (None skipped), all of them contiguous and on one
// ROCm device; None when there are none.
PyObject* require_device(PyObject*, PyObject* const* args, Py_ssize_t n) {
  const char* const kHost = "voom_amd ops need ROCm device tensors (no CPU fallback exists)";
  const char* const kStrided = "voom_amd ops need contiguous tensors";
  const char* const kOther = "all tensors must be on the same device";
  PyObject* dev = nullptr;
  std::optional<at::Device> first;
  auto fail = [&](const char* msg) -> PyObject* {
    if (msg) PyErr_SetString(PyExc_ValueError, msg);
    Py_XDECREF(dev);
    return nullptr;
  };
  try {
    for (Py_ssize_t i = 0; i < n; ++i) {
      PyObject* o = args[i];
      if (o == Py_None) continue;
      if (plain_tensor(o)) {
        const at::Tensor& t = THPVariable_Unpack(o);
        if (!t.is_cuda()) return fail(kHost);
        if (!t.is_contiguous()) return fail(kStrided);
        if (!dev) {
          first = t.device();
        } else if (first && t.device() == *first) {
          continue;
        }
      } else {
        PyObject* cuda = PyObject_GetAttrString(o, "is_cuda");
        const int is_cuda = cuda ? PyObject_IsTrue(cuda) : -1;
        Py_XDECREF(cuda);
        if (is_cuda <= 0) return fail(is_cuda < 0 ? nullptr : kHost);
        PyObject* contig = PyObject_CallMethod(o, "is_contiguous", nullptr);
        const int is_contig = contig ? PyObject_IsTrue(contig) : -1;
        Py_XDECREF(contig);
        if (is_contig <= 0) return fail(is_contig < 0 ? nullptr : kStrided);
      }
      PyObject* d = PyObject_GetAttrString(o, "device");
      if (!d) return fail(nullptr);
      if (!dev) {
        dev = d;
        continue;
      }
      const int same = PyObject_RichCompareBool(d, dev, Py_EQ);
      Py_DECREF(d);
      if (same <= 0) return fail(same < 0 ? nullptr : kOther);
    }
  } catch (const std::exception& e) {
    Py_XDECREF(dev);
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
  if (!dev) Py_RETURN_NONE;
  return dev;
}

#define VOOM_CALL(name) \
  {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&wrap<&name>)), METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {
    {"require_device", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&require_device)),
     METH_FASTCALL, nullptr},
    VOOM_CALL(voom_abi_version),
    VOOM_CALL(voom_paged_gqa_workspace_bytes),
    VOOM_CALL(voom_paged_gqa_default_splits),
    VOOM_CALL(voom_paged_gqa_decode),
    VOOM_CALL(voom_paged_gqa_noalloc_max_bytes),
    VOOM_CALL(voom_paged_gqa_decode_noalloc),
    VOOM_CALL(voom_paged_gqa_partials),
    VOOM_CALL(voom_paged_gqa_combine),
    VOOM_CALL(voom_paged_gqa_prefill_workspace_bytes),
    VOOM_CALL(voom_paged_gqa_prefill),
    VOOM_CALL(voom_merge_attn_states),
    VOOM_CALL(voom_fold_attn_state),
    VOOM_CALL(voom_mla_workspace_bytes),
    VOOM_CALL(voom_mla_absorbed_decode),
    VOOM_CALL(voom_mla_absorbed_decode_project),
    VOOM_CALL(voom_mla_sparse_workspace_bytes),
    VOOM_CALL(voom_mla_sparse_decode),
    VOOM_CALL(voom_dsa_index_scores),
    VOOM_CALL(voom_dsa_topk_workspace_bytes),
    VOOM_CALL(voom_dsa_topk),
    VOOM_CALL(voom_add_rms_norm),
    VOOM_CALL(voom_rope_split),
    VOOM_CALL(voom_silu_mul),
    VOOM_CALL(voom_gemv_bf16),
    VOOM_CALL(voom_qkv_rope_append),
    VOOM_CALL(voom_mla_head_gemv),
    VOOM_CALL(voom_mla_head_weights_bytes),
    VOOM_CALL(voom_mla_pack_head_weights),
    VOOM_CALL(voom_mla_absorb_query),
    VOOM_CALL(voom_mla_head_rows),
    VOOM_CALL(voom_lm_head_argmax),
    VOOM_CALL(voom_add_rms_norm_gemv),
    VOOM_CALL(voom_linear_rows),
    VOOM_CALL(voom_norm_swiglu_rows),
    VOOM_CALL(voom_qkv_rope_append_rows),
    VOOM_CALL(voom_position_free_workspace_bytes),
    VOOM_CALL(voom_position_free_attention),
    VOOM_CALL(voom_check_block_table),
    VOOM_CALL(voom_check_selection),
    VOOM_CALL(voom_check_position_free_pages),
    VOOM_CALL(voom_append_kv),
    VOOM_CALL(voom_gather_kv),
    VOOM_CALL(voom_append_rows),
    VOOM_CALL(voom_gather_rows),
    VOOM_CALL(voom_byteplane_split),
    VOOM_CALL(voom_byteplane_merge),
    VOOM_CALL(voom_byteplane_split_slots),
    VOOM_CALL(voom_byteplane_merge_slots),
    VOOM_CALL(voom_page_sums_verify),
    VOOM_CALL(voom_record_prepare),
    VOOM_CALL(voom_spill_record),
    VOOM_CALL(voom_reload_record),
    VOOM_CALL(voom_copy_rows),
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_calls", nullptr, -1, kMethods,
                       nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__calls() { return PyModule_Create(&kModule); }
