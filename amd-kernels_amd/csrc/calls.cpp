// The whole host side of a plain GPU call in one native function: argument
// checks, output and workspace allocation, and the launches through the C ABI.
//
// Each function takes the Python wrapper's arguments by position and either
// does the call, or, when anything about it is not the plain case (an argument
// that would be refused, CPU tensors, tensor subclasses and wrapped tensors,
// an active torch mode, a switch set in the environment), returns None without
// having done anything, and the wrapper's own checks and path follow. So every
// refusal and message stays in one place, in Python.
//
// In Python an attention call spends ~20 us on the host (checks, two or three
// allocations, five calls through ctypes) and bounds every call whose kernels
// take less. Back to back: attention on (1, 2, 256, 128) 21.2 -> 14.5 us, the
// kernels' own time; 8192 tokens into the fp8 cache 11.0 -> 4.2 us.

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/TensorSubclassLikeUtils.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/empty_like.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/version.h>

#include <climits>
#include <cstdlib>
#include <limits>

#include "../../include/moonmath_gfx950.h"

namespace {

// The launchers, by the addresses that the binding has loaded (`bind`).
struct Abi {
#define MM_ABI(X)                                                                                          \
  X(launch_v_transpose_rtne)                                                                               \
  X(moonmath_attention_forward_ex)                                                                         \
  X(moonmath_attention_forward_direct)                                                                     \
  X(moonmath_attention_direct_workspace)                                                                   \
  X(moonmath_attention_forward_lite_direct)                                                                \
  X(moonmath_attention_prefers_direct)                                                                     \
  X(moonmath_attention_plan_tail)                                                                          \
  X(moonmath_attention_vt_bytes)                                                                           \
  X(tail_workspace_bytes_rtne)                                                                             \
  X(launch_attention_forward_lite_rtne)                                                                    \
  X(launch_attention_forward_lite_rtna)                                                                    \
  X(launch_attention_forward_lite_rtz)                                                                     \
  X(lite_workspace_bytes_rtne)                                                                             \
  X(mla_decode_a16w8_multiq_workspace_for)                                                                 \
  X(moonmath_mla_effective_parts)                                                                          \
  X(moonmath_mla_slab_parts)                                                                               \
  X(launch_mla_decode_a16w8)                                                                               \
  X(launch_mla_decode_a16w8_multiq)                                                                        \
  X(launch_mla_decode_a16w8_paged_dev)                                                                     \
  X(launch_mla_decode_a16w8_multiq_paged_dev)                                                              \
  X(launch_mla_decode_a16w8_paged_blocks_dev)                                                              \
  X(launch_mla_kv_quantize)
#define MM_FIELD(name) decltype(&::name) name = nullptr;
  MM_ABI(MM_FIELD)
#undef MM_FIELD
} abi;

using at::Tensor;

// Thrown to leave a call to the Python path.
struct NotPlain {};
inline void plain(bool ok) {
  if (!ok) throw NotPlain{};
}

const Tensor& unpack(PyObject* o) {
  plain(THPVariable_CheckExact(o));
  return THPVariable_Unpack(o);
}

// A contiguous strided GPU tensor that is what it looks like.
void check_tensor(const Tensor& t, at::ScalarType dtype, c10::Device dev) {
  plain(t.defined() && t.scalar_type() == dtype && t.layout() == at::kStrided && t.device() == dev &&
        t.is_contiguous() && !at::isTensorSubclassLike(t) && !t.is_neg());
}
void check_modes() {
  plain(!c10::impl::TorchDispatchModeTLS::any_modes_set() && !at::impl::torch_function_mode_enabled());
}

int as_int(int64_t v) {
  plain(v >= INT_MIN && v <= INT_MAX);
  return (int)v;
}
int int_arg(PyObject* o) {
  plain(PyLong_CheckExact(o));
  int over = 0;
  const long v = PyLong_AsLongAndOverflow(o, &over);
  plain(over == 0);
  return as_int(v);
}
float float_arg(PyObject* o) {
  plain(PyFloat_CheckExact(o));
  return (float)PyFloat_AS_DOUBLE(o);
}
int choice(PyObject* o, const char* const* names, int n) {
  plain(PyUnicode_CheckExact(o));
  for (int i = 0; i < n; ++i)
    if (PyUnicode_CompareWithASCIIString(o, names[i]) == 0) return i;
  throw NotPlain{};
}
int mode_arg(PyObject* o) {
  static const char* const names[] = {"rtne", "rtna", "rtz"};
  return choice(o, names, 3);
}
int layout_arg(PyObject* o) {
  static const char* const names[] = {"bhsd", "bshd"};
  return choice(o, names, 2);
}

// A launcher's error code, which surfaces as the RuntimeError of the Python path.
struct LaunchFailed {
  const char* what;
  int rc;
};
void check_rc(int rc, const char* what) {
  if (rc != 0) throw LaunchFailed{what, rc};
}

void* stream_of(const Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

Tensor bytes(size_t n, const Tensor& like) {
  return at::empty({(int64_t)n}, like.options().dtype(at::kByte).requires_grad(false));
}

// Runs `body` (arguments -> what the wrapper returns); None where it is not the
// plain case. RuntimeErrors of the launchers and of the allocator pass on.
template <class Body>
PyObject* guarded(Body body) {
  HANDLE_TH_ERRORS
  try {
    return body();
  } catch (const NotPlain&) {
    Py_RETURN_NONE;
  } catch (const LaunchFailed& e) {
    return PyErr_Format(PyExc_RuntimeError, "%s returned error code %d", e.what, e.rc);
  }
  END_HANDLE_TH_ERRORS
}

struct AttnArgs {
  Tensor q, k, v, out;
  bool own_out = false;
  int B, H, Sq, Skv, mode, layout;
};

// q, k, v, out or None, round_mode, layout
AttnArgs attn_args(PyObject* q, PyObject* k, PyObject* v, PyObject* out, PyObject* mode, PyObject* layout) {
  AttnArgs a;
  a.mode = mode_arg(mode);
  a.layout = layout_arg(layout);
  a.q = unpack(q);
  a.k = unpack(k);
  a.v = unpack(v);
  plain(a.q.is_cuda());
  const auto dev = a.q.device();
  check_modes();
  for (const Tensor* t : {&a.q, &a.k, &a.v}) {
    check_tensor(*t, at::kBFloat16, dev);
    plain(t->dim() == 4);
  }
  const int sax = a.layout ? 1 : 2, hax = a.layout ? 2 : 1;
  plain(a.q.size(3) == 128 && a.k.sizes() == a.v.sizes() && a.k.size(0) == a.q.size(0) &&
        a.k.size(hax) == a.q.size(hax) && a.k.size(3) == 128);
  a.B = as_int(a.q.size(0));
  a.H = as_int(a.q.size(hax));
  a.Sq = as_int(a.q.size(sax));
  a.Skv = as_int(a.k.size(sax));
  plain(a.B > 0 && a.H > 0 && a.Sq > 0 && a.Skv > 0);
  as_int((int64_t)a.B * a.H * a.Skv);
  if (out != Py_None) {
    a.out = unpack(out);
    check_tensor(a.out, at::kBFloat16, dev);
    plain(a.out.sizes() == a.q.sizes());
    a.own_out = true;
  }
  return a;
}

// Whether the call reads V itself: a kernel that gathers V while others of its
// CTAs store `out` cannot have the two in one place, as a V_t pass before it can,
// and its 16-byte gathers want V's rows aligned, as plain loads do not.
bool direct_call(const AttnArgs& a) {
  const auto at = [](const Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()); };
  const bool apart = !a.own_out || at(a.out) + a.out.nbytes() <= at(a.v) || at(a.v) + a.v.nbytes() <= at(a.out);
  return apart && at(a.v) % 16 == 0 && abi.moonmath_attention_prefers_direct(a.B, a.H, a.Sq, a.Skv);
}

PyObject* attn_result(const AttnArgs& a, PyObject* out) {
  if (a.own_out) {
    Py_INCREF(out);
    return out;
  }
  return THPVariable_Wrap(a.out);
}

PyObject* forward(PyObject*, PyObject* const* x, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    plain(n == 6 && !std::getenv("MOONMATH_NO_TAIL") && !std::getenv("MOONMATH_FORCE_SPLIT"));
    AttnArgs a = attn_args(x[0], x[1], x[2], x[3], x[4], x[5]);
    {
      pybind11::gil_scoped_release no_gil;
      const c10::DeviceGuard guard(a.q.device());
      if (!a.own_out) a.out = at::empty_like(a.q);
      void* stream = stream_of(a.q);
      Tensor vt, ws;
      const bool direct = direct_call(a);
      size_t ws_bytes = 0;
      if (direct) {
        ws_bytes = abi.moonmath_attention_direct_workspace(a.B, a.H, a.Sq, a.Skv);
      } else {
        int plan[4];
        check_rc(abi.moonmath_attention_plan_tail(a.B, a.H, a.Sq, a.Skv, 1, 0, plan), "moonmath_attention_plan_tail");
        if (plan[3] > 0) ws_bytes = abi.tail_workspace_bytes_rtne();
        vt = bytes(abi.moonmath_attention_vt_bytes(a.B, a.H, a.Skv), a.q);
        check_rc(abi.launch_v_transpose_rtne(a.v.data_ptr(), vt.data_ptr(), a.B * a.H * a.Skv, a.Skv, a.H, a.layout,
                                             stream),
                 "launch_v_transpose");
      }
      if (ws_bytes) ws = bytes(ws_bytes, a.q);
      check_rc((direct ? abi.moonmath_attention_forward_direct : abi.moonmath_attention_forward_ex)(
                   a.q.data_ptr(), a.k.data_ptr(), direct ? a.v.data_ptr() : vt.data_ptr(), a.out.data_ptr(), a.B, a.H,
                   a.Sq, a.Skv, 128, a.layout, a.mode, ws.defined() ? ws.data_ptr() : nullptr, 0, stream),
               "launch_attention_forward");
    }
    return attn_result(a, x[3]);
  });
}

// q, k, v, read_list, write_list, threshold, phase, out or None, round_mode, layout (no must_do list)
PyObject* forward_lite(PyObject*, PyObject* const* x, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    plain(n == 10 && !std::getenv("MOONMATH_LITE_PLAIN"));
    AttnArgs a = attn_args(x[0], x[1], x[2], x[7], x[8], x[9]);
    const Tensor &read = unpack(x[3]), &write = unpack(x[4]);
    const float threshold = float_arg(x[5]);
    const int phase = int_arg(x[6]);
    const int64_t need = (int64_t)a.B * a.H * ((a.Sq + 255) / 256) * ((a.Skv + 63) / 64 + 2);
    for (const Tensor* t : {&read, &write}) {
      check_tensor(*t, at::kShort, a.q.device());
      plain(t->numel() >= need);
    }
    {
      pybind11::gil_scoped_release no_gil;
      const c10::DeviceGuard guard(a.q.device());
      if (!a.own_out) a.out = at::empty_like(a.q);
      void* stream = stream_of(a.q);
      const Tensor ws = bytes(abi.lite_workspace_bytes_rtne(a.B, a.H, a.Sq), a.q);
      if (direct_call(a)) {
        check_rc(abi.moonmath_attention_forward_lite_direct(
                     a.q.data_ptr(), a.k.data_ptr(), a.v.data_ptr(), a.out.data_ptr(), a.B, a.H, a.Sq, a.Skv, 128,
                     read.data_ptr(), write.data_ptr(), nullptr, threshold, phase, a.layout, a.mode, ws.data_ptr(),
                     stream),
                 "launch_attention_forward_lite");
      } else {
        const Tensor vt = bytes(abi.moonmath_attention_vt_bytes(a.B, a.H, a.Skv), a.q);
        check_rc(abi.launch_v_transpose_rtne(a.v.data_ptr(), vt.data_ptr(), a.B * a.H * a.Skv, a.Skv, a.H, a.layout,
                                             stream),
                 "launch_v_transpose");
        const auto launch = a.mode == 0   ? abi.launch_attention_forward_lite_rtne
                            : a.mode == 1 ? abi.launch_attention_forward_lite_rtna
                                          : abi.launch_attention_forward_lite_rtz;
        check_rc(launch(a.q.data_ptr(), a.k.data_ptr(), vt.data_ptr(), a.out.data_ptr(), a.B, a.H, a.Sq, a.Skv, 128,
                        read.data_ptr(), write.data_ptr(), nullptr, threshold, phase, a.layout, ws.data_ptr(), stream),
                 "launch_attention_forward_lite");
      }
    }
    return attn_result(a, x[7]);
  });
}

struct MlaArgs {
  Tensor q_lat, q_pe, o_lat;
  int B, H, q_len;
};

MlaArgs mla_args(PyObject* q_lat, PyObject* q_pe, PyObject* o_lat, bool multiq) {
  MlaArgs a{unpack(q_lat), unpack(q_pe), unpack(o_lat), 0, 0, 1};
  plain(a.q_lat.is_cuda());
  check_modes();
  for (const Tensor* t : {&a.q_lat, &a.q_pe, &a.o_lat}) check_tensor(*t, at::kBFloat16, a.q_lat.device());
  const int64_t D = a.q_lat.dim();
  plain((D == 4 || (D == 3 && !multiq)) && a.q_pe.dim() == D && a.o_lat.sizes() == a.q_lat.sizes());
  plain(a.q_lat.size(D - 1) == 512 && a.q_pe.size(D - 1) == 64 &&
        a.q_pe.sizes().slice(0, D - 1) == a.q_lat.sizes().slice(0, D - 1));
  a.B = as_int(a.q_lat.size(0));
  a.H = as_int(a.q_lat.size(D - 2));
  if (D == 4) a.q_len = as_int(a.q_lat.size(1));
  plain(a.B >= 1 && a.H >= 1 && a.H <= 128 && a.q_len >= (multiq ? 2 : 1) && a.q_len <= 8);
  return a;
}

Tensor mla_workspace(const MlaArgs& a, int parts) {
  const int eff = abi.moonmath_mla_effective_parts(a.B, a.H, parts, a.q_len, 1);
  return eff <= 1 ? Tensor() : bytes(abi.mla_decode_a16w8_multiq_workspace_for(a.B, a.H, eff, a.q_len), a.q_lat);
}

const Tensor& index_tensor(PyObject* o, const Tensor& q, int64_t least) {
  const Tensor& t = unpack(o);
  check_tensor(t, at::kInt, q.device());
  plain(t.numel() >= least);
  return t;
}

void* ptr_or_null(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

// The single-query ops take scale_p and use it nowhere, but refuse what is no number.
void unused_scale_p(PyObject* o, bool multiq) {
  if (!multiq) float_arg(o);
}

// q_lat, q_pe, kv, o_lat, scale, kv_scale, scale_p, multiq
PyObject* mla_slab(PyObject*, PyObject* const* x, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    plain(n == 8);
    const bool multiq = x[7] == Py_True;
    unused_scale_p(x[6], multiq);
    const MlaArgs a = mla_args(x[0], x[1], x[3], multiq);
    plain(multiq || a.q_len == 1);
    const Tensor& kv = unpack(x[2]);
    check_tensor(kv, at::kFloat8_e4m3fn, a.q_lat.device());
    plain(kv.dim() == 3 && kv.size(2) == 576 && kv.size(0) == a.B && kv.size(1) >= 1);
    const int S = as_int(kv.size(1));
    const float scale = float_arg(x[4]), kv_scale = float_arg(x[5]);
    {
      pybind11::gil_scoped_release no_gil;
      const c10::DeviceGuard guard(a.q_lat.device());
      const int parts = abi.moonmath_mla_slab_parts(a.B, a.H, S, a.q_len);
      const Tensor ws = mla_workspace(a, parts);
      void* stream = stream_of(a.q_lat);
      if (multiq)
        check_rc(abi.launch_mla_decode_a16w8_multiq(a.q_lat.data_ptr(), a.q_pe.data_ptr(), kv.data_ptr(),
                                                    a.o_lat.data_ptr(), a.B, a.H, S, a.q_len, 512, 64, scale, kv_scale,
                                                    ptr_or_null(ws), stream),
                 "launch_mla_decode_a16w8_multiq");
      else
        check_rc(abi.launch_mla_decode_a16w8(a.q_lat.data_ptr(), a.q_pe.data_ptr(), kv.data_ptr(), nullptr,
                                             a.o_lat.data_ptr(), a.B, a.H, S, 512, 64, scale, kv_scale, 1.0f,
                                             ptr_or_null(ws), stream),
                 "launch_mla_decode_a16w8");
    }
    Py_RETURN_TRUE;
  });
}

// q_lat, q_pe, kv_pool, o_lat, seq_lens, rows or None, kv_indices, kv_indptr, parts, scale, kv_scale, scale_p, multiq
PyObject* mla_paged(PyObject*, PyObject* const* x, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    plain(n == 13);
    const bool multiq = x[12] == Py_True;
    unused_scale_p(x[11], multiq);
    const MlaArgs a = mla_args(x[0], x[1], x[3], multiq);
    const Tensor& pool = unpack(x[2]);
    check_tensor(pool, at::kFloat8_e4m3fn, a.q_lat.device());
    plain(pool.dim() >= 1 && pool.size(-1) == 576);
    const Tensor& lens = index_tensor(x[4], a.q_lat, a.B);
    const Tensor rows = x[5] == Py_None ? Tensor() : index_tensor(x[5], a.q_lat, a.B);
    const Tensor& indices = index_tensor(x[6], a.q_lat, 0);
    const Tensor& indptr = index_tensor(x[7], a.q_lat, a.B + 1);
    const int parts = int_arg(x[8]);
    plain(parts <= (1 << 20));
    const float scale = float_arg(x[9]), kv_scale = float_arg(x[10]);
    const size_t kv_bytes = (size_t)indices.numel() * 576;
    {
      pybind11::gil_scoped_release no_gil;
      const c10::DeviceGuard guard(a.q_lat.device());
      const Tensor ws = mla_workspace(a, parts);
      void* stream = stream_of(a.q_lat);
      if (multiq)
        check_rc(abi.launch_mla_decode_a16w8_multiq_paged_dev(
                     a.q_lat.data_ptr(), a.q_pe.data_ptr(), pool.data_ptr(), a.o_lat.data_ptr(), lens.data_ptr(),
                     ptr_or_null(rows), indices.data_ptr(), indptr.data_ptr(), a.B, a.H, parts, a.q_len, 512, 64,
                     scale, kv_scale, ptr_or_null(ws), stream, kv_bytes),
                 "launch_mla_decode_a16w8_multiq_paged_dev");
      else
        check_rc(abi.launch_mla_decode_a16w8_paged_dev(
                     a.q_lat.data_ptr(), a.q_pe.data_ptr(), pool.data_ptr(), a.o_lat.data_ptr(), lens.data_ptr(),
                     ptr_or_null(rows), indices.data_ptr(), indptr.data_ptr(), a.B, a.H, parts, 512, 64, scale,
                     kv_scale, 1.0f, ptr_or_null(ws), stream, kv_bytes, a.q_len),
                 "launch_mla_decode_a16w8_paged_dev");
    }
    Py_RETURN_TRUE;
  });
}

// q_lat, q_pe, kv_pool, o_lat, seq_lens, block_table, parts, scale, kv_scale, scale_p, rows or None
PyObject* mla_blocks(PyObject*, PyObject* const* x, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    plain(n == 11);
    unused_scale_p(x[9], false);
    const MlaArgs a = mla_args(x[0], x[1], x[3], false);
    const Tensor& pool = unpack(x[2]);
    check_tensor(pool, at::kFloat8_e4m3fn, a.q_lat.device());
    plain(pool.dim() >= 1 && pool.size(-1) == 576 && pool.numel() % (64 * 576) == 0);
    const Tensor& lens = index_tensor(x[4], a.q_lat, a.B);
    const Tensor& table = index_tensor(x[5], a.q_lat, 1);
    plain(table.dim() == 2 && table.size(0) == a.B && table.size(1) >= 1);
    const Tensor rows = x[10] == Py_None ? Tensor() : index_tensor(x[10], a.q_lat, a.B);
    const int parts = int_arg(x[6]);
    plain(parts <= (1 << 20));
    const float scale = float_arg(x[7]), kv_scale = float_arg(x[8]);
    const int max_blocks = as_int(table.size(1)), num_blocks = as_int(pool.numel() / (64 * 576));
    {
      pybind11::gil_scoped_release no_gil;
      const c10::DeviceGuard guard(a.q_lat.device());
      const Tensor ws = mla_workspace(a, parts);
      check_rc(abi.launch_mla_decode_a16w8_paged_blocks_dev(
                   a.q_lat.data_ptr(), a.q_pe.data_ptr(), pool.data_ptr(), a.o_lat.data_ptr(), lens.data_ptr(),
                   ptr_or_null(rows), table.data_ptr(), max_blocks, num_blocks, a.B, a.H, parts, a.q_len, 512, 64,
                   scale, kv_scale, 1.0f, ptr_or_null(ws), table.data_ptr(), stream_of(a.q_lat)),
               "launch_mla_decode_a16w8_paged_blocks_dev");
    }
    Py_RETURN_TRUE;
  });
}

// c_kv, k_pe, kv_pool, slots, kv_scale, saturate
PyObject* kv_quantize(PyObject*, PyObject* const* x, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    plain(n == 6 && PyBool_Check(x[5]));
    const Tensor &c_kv = unpack(x[0]), &k_pe = unpack(x[1]), &pool = unpack(x[2]), &slots = unpack(x[3]);
    plain(c_kv.is_cuda());
    check_modes();
    const auto dev = c_kv.device();
    check_tensor(c_kv, at::kBFloat16, dev);
    check_tensor(k_pe, at::kBFloat16, dev);
    check_tensor(pool, at::kFloat8_e4m3fn, dev);
    check_tensor(slots, at::kInt, dev);
    plain(c_kv.dim() >= 1 && c_kv.size(-1) == 512 && k_pe.dim() >= 1 && k_pe.size(-1) == 64 && pool.dim() >= 1 &&
          pool.size(-1) == 576);
    const int64_t N = c_kv.numel() / 512;
    plain(k_pe.numel() / 64 == N && slots.numel() == N);
    plain(PyFloat_CheckExact(x[4]));
    const double scale = PyFloat_AS_DOUBLE(x[4]);
    plain(scale > 0.0 && scale < std::numeric_limits<double>::infinity());
    const int saturate = x[5] == Py_True;
    {
      pybind11::gil_scoped_release no_gil;
      const c10::DeviceGuard guard(dev);
      check_rc(abi.launch_mla_kv_quantize(c_kv.data_ptr(), k_pe.data_ptr(), pool.data_ptr(), slots.data_ptr(), N,
                                          pool.numel() / 576, (float)scale, saturate, stream_of(c_kv)),
               "launch_mla_kv_quantize");
    }
    Py_RETURN_TRUE;
  });
}

// bind({name: address}): the loaded library's launchers.
PyObject* bind(PyObject*, PyObject* table) {
#define MM_BIND(name)                                                            \
  {                                                                              \
    PyObject* v = PyDict_GetItemString(table, #name);                            \
    if (!v) {                                                                    \
      PyErr_SetString(PyExc_KeyError, #name);                                    \
      return nullptr;                                                            \
    }                                                                            \
    abi.name = reinterpret_cast<decltype(abi.name)>(PyLong_AsVoidPtr(v));        \
    if (PyErr_Occurred()) return nullptr;                                        \
  }
  MM_ABI(MM_BIND)
#undef MM_BIND
  Py_RETURN_NONE;
}

PyObject* bound_names(PyObject*, PyObject*) {
#define MM_NAME(name) #name,
  static const char* const names[] = {MM_ABI(MM_NAME)};
#undef MM_NAME
  PyObject* t = PyTuple_New(sizeof(names) / sizeof(names[0]));
  if (!t) return nullptr;
  for (size_t i = 0; i < sizeof(names) / sizeof(names[0]); ++i) PyTuple_SET_ITEM(t, i, PyUnicode_FromString(names[i]));
  return t;
}

PyObject* torch_version(PyObject*, PyObject*) { return PyUnicode_FromString(TORCH_VERSION); }

#define MM_FAST(name) {#name, (PyCFunction)(void (*)())name, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {MM_FAST(forward),
                         MM_FAST(forward_lite),
                         MM_FAST(mla_slab),
                         MM_FAST(mla_paged),
                         MM_FAST(mla_blocks),
                         MM_FAST(kv_quantize),
                         {"bind", bind, METH_O, nullptr},
                         {"bound_names", bound_names, METH_NOARGS, nullptr},
                         {"torch_version", torch_version, METH_NOARGS, nullptr},
                         {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_calls", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__calls() { return PyModule_Create(&module); }
