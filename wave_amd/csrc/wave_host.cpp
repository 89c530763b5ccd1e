// The host side of one operator call in native code: checks, scratch, stream and outputs for the calls that the
// Python wrappers of wave_amd/mxfp4.py would make through ctypes (their counterpart in the reference is native as
// well: wave_lang/kernel/wave/runtime/runtime.cpp:123-203).
//
// What bounds small problems is this path: with the checks in Python and ctypes in between, a call took the host
// 9.9 us (mxfp4_gemm) and 10.7 us (quantize_mxfp4, two outputs) while the kernels of a decode projection take
// 3.5 + 7.4 us.  Here: 4.5 and 5.0 us, of which the launch is about 3; the five calls of an expert MLP 75 -> 27 us.
//
// Every function here serves the common form of a call (contiguous tensors of the right shapes on the current
// device, the library's own scratch) and reports with None / False that it launched nothing for anything else: the
// wrapper then runs its own checks, which raise the errors, copy what is not contiguous and grow the scratch.  The
// entry points of the C ABI are handed over as addresses by the loader, so that the library it loaded is the one called.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ops/empty.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>

#include <map>
#include <tuple>
#include <unordered_map>

#include "../../include/wave_mxfp4.h"

namespace {

struct Entry {
  decltype(&wave_mxfp4_gemm) gemm = nullptr;
  decltype(&wave_mxfp4_workspace_bytes) workspace_bytes = nullptr;
  decltype(&wave_mxfp4_gemm_grouped) grouped = nullptr;
  decltype(&wave_mxfp4_grouped_workspace_bytes) grouped_workspace_bytes = nullptr;
  decltype(&wave_mxfp4_gemm_gated_quantize) gated = nullptr;
  decltype(&wave_mxfp8_gemm) mxfp8 = nullptr;
  decltype(&wave_mxfp8_gemm_b_preshuffled) mxfp8_b = nullptr;
  decltype(&wave_mxfp8_workspace_bytes) mxfp8_workspace_bytes = nullptr;
  decltype(&wave_mxfp4_quantize) quantize = nullptr;
  decltype(&wave_mxfp4_quantize_rows) quantize_rows = nullptr;
  decltype(&wave_mxfp4_moe_align_block_size) moe_align = nullptr;
  decltype(&wave_mxfp4_silu_and_mul_quantize) silu_quantize = nullptr;
} g_entry;

// (device, stream) -> scratch the wrapper allocated for it.  The wrapper never frees a buffer it has handed out, so an
// address read here stays valid; both tables are only touched under the GIL.
struct Scratch {
  void *ptr = nullptr;
  size_t bytes = 0;
};
std::map<std::pair<int, void *>, Scratch> g_scratch;
// scratch bytes of a dense problem: the library prices every tile shape to answer
std::map<std::tuple<int64_t, int64_t, int64_t, int, int>, size_t> g_bytes;
constexpr size_t kMaxPlans = 4096;

const at::Tensor *tensor(PyObject *o) { return THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr; }

// The current device if `t` is a GPU tensor, else one that no tensor is on (without a GPU there is none to ask for)
int device_for(const at::Tensor *t) { return t->is_cuda() ? (int)c10::hip::current_device() : -2; }

// A contiguous GPU tensor on device `dev`
bool on_gpu(const at::Tensor *t, int dev) { return t->is_cuda() && t->get_device() == dev && t->is_contiguous(); }

bool bytes_on_gpu(const at::Tensor *t, int dev) {
  return (t->scalar_type() == at::kByte || t->scalar_type() == at::kChar) && on_gpu(t, dev);
}

bool ints_on_gpu(const at::Tensor *t, int dev) { return t->scalar_type() == at::kInt && on_gpu(t, dev); }

int out_code(const at::Tensor *t) {
  return t->scalar_type() == at::kBFloat16 ? WAVE_MXFP4_OUT_BF16 : t->scalar_type() == at::kFloat ? WAVE_MXFP4_OUT_F32 : -1;
}

int in_code(const at::Tensor *t) {
  switch (t->scalar_type()) {
    case at::kFloat: return WAVE_MXFP4_IN_F32;
    case at::kBFloat16: return WAVE_MXFP4_IN_BF16;
    case at::kHalf: return WAVE_MXFP4_IN_F16;
    default: return -1;
  }
}

int64_t padded_scale_bytes(int64_t rows, int64_t ks) { return (rows + 31) / 32 * 32 * ((ks + 7) / 8 * 8); }

bool scales_ok(const at::Tensor *s, int64_t rows, int64_t ks, int layout) {
  switch (layout) {
    case WAVE_MXFP4_SCALE_ROW_MAJOR: return s->dim() == 2 && s->size(0) == rows && s->size(1) == ks;
    case WAVE_MXFP4_SCALE_PER_ROW: return s->dim() == 1 && s->size(0) == rows;
    case WAVE_MXFP4_SCALE_E8M0_SHUFFLE:
    case WAVE_MXFP4_SCALE_MFMA32: return s->numel() >= padded_scale_bytes(rows, ks);
    default: return false;
  }
}

// The scratch of the current stream if it holds `bytes` (null and true where none is needed)
bool scratch_for(int dev, void *stream, size_t bytes, Scratch &out) {
  out = Scratch{};
  if (bytes == 0) return true;
  const auto it = g_scratch.find({dev, stream});
  if (it == g_scratch.end() || it->second.bytes < bytes) return false;
  out = {it->second.ptr, bytes};
  return true;
}

void *current_stream(int dev) { return (void *)c10::hip::getCurrentHIPStream((c10::DeviceIndex)dev).stream(); }

// One call into the library, without the GIL as ctypes would make it
template <class F, class... A>
int call(F f, A... a) {
  int st;
  Py_BEGIN_ALLOW_THREADS st = f(a...);
  Py_END_ALLOW_THREADS return st;
}

at::Tensor new_bytes(int64_t r, int64_t c, int dev) {
  return at::empty({r, c}, at::TensorOptions().dtype(at::kByte).device(at::kCUDA, (c10::DeviceIndex)dev));
}

at::Tensor new_scales(int64_t rows, int64_t ks, int layout, int dev) {
  return layout == WAVE_MXFP4_SCALE_ROW_MAJOR ? new_bytes(rows, ks, dev)
                                              : new_bytes((rows + 31) / 32 * 32, (ks + 7) / 8 * 8, dev);
}

PyObject *pair(at::Tensor a, at::Tensor b) {
  PyObject *t = PyTuple_New(2);
  if (!t) return nullptr;
  PyTuple_SET_ITEM(t, 0, THPVariable_Wrap(std::move(a)));
  PyTuple_SET_ITEM(t, 1, THPVariable_Wrap(std::move(b)));
  return t;
}

int to_int(PyObject *o) { return (int)PyLong_AsLong(o); }

#define WAVE_DECLINE_BOOL Py_RETURN_FALSE
#define WAVE_DECLINE Py_RETURN_NONE

// gemm(x, x_scales, w_t, w_scales, out, a_scale_layout, b_scale_layout, b_layout, split_k, variant) -> launched
PyObject *host_gemm(PyObject *, PyObject *const *v, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  if (n_args != 10 || !g_entry.gemm) WAVE_DECLINE_BOOL;
  const at::Tensor *x = tensor(v[0]), *xs = tensor(v[1]), *w = tensor(v[2]), *ws = tensor(v[3]), *out = tensor(v[4]);
  if (!x || !xs || !w || !ws || !out || x->dim() != 2 || w->dim() != 2 || out->dim() != 2) WAVE_DECLINE_BOOL;
  const int dev = device_for(x);
  if (!bytes_on_gpu(x, dev) || !bytes_on_gpu(xs, dev) || !bytes_on_gpu(w, dev) || !bytes_on_gpu(ws, dev) || !on_gpu(out, dev))
    WAVE_DECLINE_BOOL;
  int asl = to_int(v[5]);
  const int bsl = to_int(v[6]), bl = to_int(v[7]), split = to_int(v[8]), variant = to_int(v[9]), od = out_code(out);
  if (PyErr_Occurred()) return nullptr;
  if (asl == WAVE_MXFP4_SCALE_ROW_MAJOR && xs->dim() == 1) asl = WAVE_MXFP4_SCALE_PER_ROW;
  const int64_t m = x->size(0), kp = x->size(1), n = w->size(0), k = 2 * kp;
  if (m == 0 || n == 0 || k == 0 || k % 32 != 0 || w->size(1) != kp || od < 0 || out->size(0) != m || out->size(1) != n ||
      !scales_ok(xs, m, k / 32, asl) || !scales_ok(ws, n, k / 32, bsl))
    WAVE_DECLINE_BOOL;
  const auto key = std::make_tuple(m, n, k, split, variant);
  auto it = g_bytes.find(key);
  if (it == g_bytes.end()) {
    if (g_bytes.size() >= kMaxPlans) g_bytes.clear();
    it = g_bytes.emplace(key, g_entry.workspace_bytes(m, n, k, split, variant)).first;
  }
  void *stream = current_stream(dev);
  Scratch s;
  if (!scratch_for(dev, stream, it->second, s)) WAVE_DECLINE_BOOL;
  const int st = call(g_entry.gemm, x->const_data_ptr(), xs->const_data_ptr(), w->const_data_ptr(), ws->const_data_ptr(),
                      out->mutable_data_ptr(), m, n, k, od, asl, bsl, bl, split, s.ptr, s.bytes, variant, stream);
  return PyBool_FromLong(st == WAVE_MXFP4_OK);
  END_HANDLE_TH_ERRORS
}

// grouped(x, x_scales, w_t, w_scales, offsets, out, a_scale_layout, b_scale_layout, b_layout, variant) -> launched
PyObject *host_grouped(PyObject *, PyObject *const *v, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  if (n_args != 10 || !g_entry.grouped) WAVE_DECLINE_BOOL;
  const at::Tensor *x = tensor(v[0]), *xs = tensor(v[1]), *w = tensor(v[2]), *ws = tensor(v[3]), *offs = tensor(v[4]), *out = tensor(v[5]);
  if (!x || !xs || !w || !ws || !offs || !out || x->dim() != 2 || w->dim() != 3 || out->dim() != 2) WAVE_DECLINE_BOOL;
  const int dev = device_for(x);
  if (!bytes_on_gpu(x, dev) || !bytes_on_gpu(xs, dev) || !bytes_on_gpu(w, dev) || !bytes_on_gpu(ws, dev) ||
      !ints_on_gpu(offs, dev) || !on_gpu(out, dev))
    WAVE_DECLINE_BOOL;
  const int asl = to_int(v[6]), bsl = to_int(v[7]), bl = to_int(v[8]), variant = to_int(v[9]), od = out_code(out);
  if (PyErr_Occurred()) return nullptr;
  const int64_t rows = x->size(0), kp = x->size(1), e = w->size(0), n = w->size(1), k = 2 * kp, ks = k / 32;
  const bool ws_ok = bsl == WAVE_MXFP4_SCALE_ROW_MAJOR ? ws->dim() == 3 && ws->size(0) == e && ws->size(1) == n && ws->size(2) == ks
                                                       : ws->numel() >= e * padded_scale_bytes(n, ks);
  if (rows == 0 || n == 0 || k == 0 || e == 0 || k % 32 != 0 || w->size(2) != kp || offs->numel() != e + 1 || od < 0 ||
      out->size(0) != rows || out->size(1) != n || asl == WAVE_MXFP4_SCALE_PER_ROW || !scales_ok(xs, rows, ks, asl) || !ws_ok)
    WAVE_DECLINE_BOOL;
  void *stream = current_stream(dev);
  Scratch s;
  if (!scratch_for(dev, stream, g_entry.grouped_workspace_bytes(rows, n, k, (int)e), s)) WAVE_DECLINE_BOOL;
  const int st = call(g_entry.grouped, x->const_data_ptr(), xs->const_data_ptr(), w->const_data_ptr(), ws->const_data_ptr(),
                      out->mutable_data_ptr(), (const int32_t *)offs->const_data_ptr(), (int)e, rows, n, k, od, asl, bsl, bl,
                      variant, s.ptr, s.bytes, stream);
  return PyBool_FromLong(st == WAVE_MXFP4_OK);
  END_HANDLE_TH_ERRORS
}

// gated(x, x_scales, w_il, w_scales_il, offsets or None, a_scale_layout, b_scale_layout, act_scale_layout)
//   -> (q, scales), the status if the library refused the problem, or None
PyObject *host_gated(PyObject *, PyObject *const *v, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  if (n_args != 8 || !g_entry.gated) WAVE_DECLINE;
  const bool grouped = v[4] != Py_None;
  const at::Tensor *x = tensor(v[0]), *xs = tensor(v[1]), *w = tensor(v[2]), *ws = tensor(v[3]), *offs = grouped ? tensor(v[4]) : nullptr;
  if (!x || !xs || !w || !ws || (grouped && !offs) || x->dim() != 2 || w->dim() != (grouped ? 3 : 2)) WAVE_DECLINE;
  const int dev = device_for(x);
  if (!bytes_on_gpu(x, dev) || !bytes_on_gpu(xs, dev) || !bytes_on_gpu(w, dev) || !bytes_on_gpu(ws, dev) ||
      (grouped && !ints_on_gpu(offs, dev)))
    WAVE_DECLINE;
  const int asl = to_int(v[5]), bsl = to_int(v[6]), actl = to_int(v[7]);
  if (PyErr_Occurred()) return nullptr;
  const int64_t rows = x->size(0), kp = x->size(1), e = grouped ? w->size(0) : 0, n = w->size(-2), k = 2 * kp;
  // (the wrapper does not check the size of the interleaved scales either: the library's own checks are what there is)
  if (rows == 0 || n == 0 || k == 0 || k % 32 != 0 || n % 64 != 0 || w->size(-1) != kp || (grouped && (e == 0 || offs->numel() != e + 1)) ||
      actl < 0 || actl > WAVE_MXFP4_SCALE_MFMA32 || !scales_ok(xs, rows, k / 32, asl))
    WAVE_DECLINE;
  void *stream = current_stream(dev);
  Scratch s;
  if (!scratch_for(dev, stream, g_entry.grouped_workspace_bytes(rows, n, k, (int)(e > 1 ? e : 1)), s)) WAVE_DECLINE;
  const int64_t inter = n / 2;
  at::Tensor q = new_bytes(rows, inter / 2, dev), sc = new_scales(rows, inter / 32, actl, dev);
  const int st = call(g_entry.gated, x->const_data_ptr(), xs->const_data_ptr(), w->const_data_ptr(), ws->const_data_ptr(),
                      q.mutable_data_ptr(), sc.mutable_data_ptr(), grouped ? (const int32_t *)offs->const_data_ptr() : nullptr,
                      (int)e, rows, n, k, asl, bsl, actl, s.ptr, s.bytes, stream);
  if (st != WAVE_MXFP4_OK) return PyLong_FromLong(st);
  return pair(std::move(q), std::move(sc));
  END_HANDLE_TH_ERRORS
}

// An MXFP8 operand's format from its dtype and the format the caller named (-1: none); -1: not served here
int fp8_format(const at::Tensor *t, int named) {
  switch (t->scalar_type()) {
    case at::kFloat8_e4m3fn: return named < 0 || named == WAVE_MXFP8_E4M3 ? WAVE_MXFP8_E4M3 : -1;
    case at::kFloat8_e5m2: return named < 0 || named == WAVE_MXFP8_E5M2 ? WAVE_MXFP8_E5M2 : -1;
    case at::kByte:
    case at::kChar: return named < 0 ? WAVE_MXFP8_E5M2 : named;
    default: return -1;
  }
}

// mxfp8(x, x_scales, w_t, w_scales, out, x_format, w_format, variant, b_preshuffled, a_scale_layout, b_scale_layout)
//   -> launched
PyObject *host_mxfp8(PyObject *, PyObject *const *v, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  if (n_args != 11 || !g_entry.mxfp8 || !g_entry.mxfp8_b) WAVE_DECLINE_BOOL;
  const at::Tensor *x = tensor(v[0]), *xs = tensor(v[1]), *w = tensor(v[2]), *ws = tensor(v[3]), *out = tensor(v[4]);
  if (!x || !xs || !w || !ws || !out || x->dim() != 2 || w->dim() != 2 || out->dim() != 2) WAVE_DECLINE_BOOL;
  const int dev = device_for(x);
  if (!on_gpu(x, dev) || !bytes_on_gpu(xs, dev) || !on_gpu(w, dev) || !bytes_on_gpu(ws, dev) || !on_gpu(out, dev)) WAVE_DECLINE_BOOL;
  const int fa = fp8_format(x, to_int(v[5])), fb = fp8_format(w, to_int(v[6])), variant = to_int(v[7]);
  const bool pre = PyObject_IsTrue(v[8]) == 1;
  const int asl = to_int(v[9]), bsl = to_int(v[10]), od = out_code(out);
  if (PyErr_Occurred()) return nullptr;
  const bool x4 = fa == WAVE_MXFP8_E2M1, w4 = fb == WAVE_MXFP8_E2M1;
  const int64_t m = x->size(0), n = w->size(0), k = x4 ? 2 * x->size(1) : x->size(1);
  if (fa < 0 || fb < 0 || (x4 && w4) || m == 0 || n == 0 || k == 0 || k % 128 != 0 || w->size(1) != (w4 ? k / 2 : k) || od < 0 ||
      out->size(0) != m || out->size(1) != n || (!pre && (asl != WAVE_MXFP4_SCALE_ROW_MAJOR || bsl != WAVE_MXFP4_SCALE_ROW_MAJOR)) ||
      !scales_ok(xs, m, k / 32, asl) || !scales_ok(ws, n, k / 32, bsl))
    WAVE_DECLINE_BOOL;
  void *stream = current_stream(dev);
  Scratch s;
  if (!scratch_for(dev, stream, g_entry.mxfp8_workspace_bytes(m, n, k), s)) WAVE_DECLINE_BOOL;
  const int st = pre ? call(g_entry.mxfp8_b, x->const_data_ptr(), xs->const_data_ptr(), w->const_data_ptr(), ws->const_data_ptr(),
                            out->mutable_data_ptr(), m, n, k, fa, fb, od, asl, bsl, s.ptr, s.bytes, stream)
                     : call(g_entry.mxfp8, x->const_data_ptr(), xs->const_data_ptr(), w->const_data_ptr(), ws->const_data_ptr(),
                            out->mutable_data_ptr(), m, n, k, fa, fb, od, s.ptr, s.bytes, variant, stream);
  return PyBool_FromLong(st == WAVE_MXFP4_OK);
  END_HANDLE_TH_ERRORS
}

// quantize(x, scale_layout) -> (q, scales) or None
PyObject *host_quantize(PyObject *, PyObject *const *v, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  if (n_args != 2 || !g_entry.quantize) WAVE_DECLINE;
  const at::Tensor *x = tensor(v[0]);
  if (!x || x->dim() != 2) WAVE_DECLINE;
  const int dev = device_for(x), dt = in_code(x), layout = to_int(v[1]);
  if (PyErr_Occurred()) return nullptr;
  const int64_t rows = x->size(0), k = x->size(1);
  if (dt < 0 || !on_gpu(x, dev) || rows == 0 || k == 0 || k % 32 != 0 || layout < 0 || layout > WAVE_MXFP4_SCALE_MFMA32) WAVE_DECLINE;
  at::Tensor q = new_bytes(rows, k / 2, dev), s = new_scales(rows, k / 32, layout, dev);
  if (call(g_entry.quantize, x->const_data_ptr(), dt, q.mutable_data_ptr(), s.mutable_data_ptr(), rows, k, layout,
           current_stream(dev)) != WAVE_MXFP4_OK)
    WAVE_DECLINE;
  return pair(std::move(q), std::move(s));
  END_HANDLE_TH_ERRORS
}

// quantize_rows(x, row_ids, row_div, scale_layout) -> (q, scales) or None
PyObject *host_quantize_rows(PyObject *, PyObject *const *v, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  if (n_args != 4 || !g_entry.quantize_rows) WAVE_DECLINE;
  const at::Tensor *x = tensor(v[0]), *ids = tensor(v[1]);
  if (!x || !ids || x->dim() != 2 || ids->dim() != 1) WAVE_DECLINE;
  const int dev = device_for(x), dt = in_code(x), div = to_int(v[2]), layout = to_int(v[3]);
  if (PyErr_Occurred()) return nullptr;
  const int64_t src = x->size(0), k = x->size(1), rows = ids->numel();
  if (dt < 0 || !on_gpu(x, dev) || !ints_on_gpu(ids, dev) || rows == 0 || k == 0 || k % 32 != 0 || layout < 0 ||
      layout > WAVE_MXFP4_SCALE_MFMA32)
    WAVE_DECLINE;
  at::Tensor q = new_bytes(rows, k / 2, dev), s = new_scales(rows, k / 32, layout, dev);
  if (call(g_entry.quantize_rows, x->const_data_ptr(), dt, src, (const int32_t *)ids->const_data_ptr(), div, q.mutable_data_ptr(),
           s.mutable_data_ptr(), rows, k, layout, current_stream(dev)) != WAVE_MXFP4_OK)
    WAVE_DECLINE;
  return pair(std::move(q), std::move(s));
  END_HANDLE_TH_ERRORS
}

// moe_align(topk_ids, num_experts, block_size, sorted_ids, expert_ids, num_tokens_post_pad, expert_offsets or None)
//   -> launched
PyObject *host_moe_align(PyObject *, PyObject *const *v, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  if (n_args != 7 || !g_entry.moe_align) WAVE_DECLINE_BOOL;
  const at::Tensor *ids = tensor(v[0]), *sorted = tensor(v[3]), *experts = tensor(v[4]), *total = tensor(v[5]);
  const at::Tensor *offs = v[6] == Py_None ? nullptr : tensor(v[6]);
  if (!ids || !sorted || !experts || !total || (v[6] != Py_None && !offs)) WAVE_DECLINE_BOOL;
  const int dev = device_for(ids);
  const bool wide = ids->scalar_type() == at::kLong;
  const long ne = PyLong_AsLong(v[1]), bs = PyLong_AsLong(v[2]);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    WAVE_DECLINE_BOOL;
  }
  if ((!wide && ids->scalar_type() != at::kInt) || !on_gpu(ids, dev) || !ints_on_gpu(sorted, dev) || !ints_on_gpu(experts, dev) ||
      !ints_on_gpu(total, dev) || total->numel() < 1 || ne < 1 || ne > 65536 || bs < 1 || bs > 0x7FFFFFFF ||
      (offs && (!ints_on_gpu(offs, dev) || offs->numel() < ne + 1)))
    WAVE_DECLINE_BOOL;
  const int st = call(g_entry.moe_align, ids->const_data_ptr(), wide ? 1 : 0, ids->numel(), (int)ne, (int)bs,
                      (int32_t *)sorted->mutable_data_ptr(), sorted->numel(), (int32_t *)experts->mutable_data_ptr(),
                      experts->numel(), (int32_t *)total->mutable_data_ptr(),
                      offs ? (int32_t *)offs->mutable_data_ptr() : nullptr, current_stream(dev));
  return PyBool_FromLong(st == WAVE_MXFP4_OK);
  END_HANDLE_TH_ERRORS
}

// silu_quantize(gate, up, scale_layout) -> (q, scales) or None
PyObject *host_silu_quantize(PyObject *, PyObject *const *v, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  if (n_args != 3 || !g_entry.silu_quantize) WAVE_DECLINE;
  const at::Tensor *gate = tensor(v[0]), *up = tensor(v[1]);
  if (!gate || !up || gate->dim() != 2 || up->dim() != 2) WAVE_DECLINE;
  const int dev = device_for(gate), dt = in_code(gate), layout = to_int(v[2]);
  if (PyErr_Occurred()) return nullptr;
  const int64_t rows = gate->size(0), n = gate->size(1);
  if ((dt != WAVE_MXFP4_IN_BF16 && dt != WAVE_MXFP4_IN_F16) || up->scalar_type() != gate->scalar_type() || !gate->is_cuda() ||
      gate->get_device() != dev || !up->is_cuda() || up->get_device() != dev || up->size(0) != rows || up->size(1) != n || rows == 0 ||
      n == 0 || n % 32 != 0 || gate->stride(1) != 1 || up->stride(1) != 1 || layout < 0 || layout > WAVE_MXFP4_SCALE_MFMA32)
    WAVE_DECLINE;
  at::Tensor q = new_bytes(rows, n / 2, dev), s = new_scales(rows, n / 32, layout, dev);
  if (call(g_entry.silu_quantize, gate->const_data_ptr(), up->const_data_ptr(), gate->stride(0), up->stride(0), dt,
           q.mutable_data_ptr(), s.mutable_data_ptr(), rows, n, layout, current_stream(dev)) != WAVE_MXFP4_OK)
    WAVE_DECLINE;
  return pair(std::move(q), std::move(s));
  END_HANDLE_TH_ERRORS
}

// set_scratch(device, stream, address, bytes): the wrapper's buffer for that stream
PyObject *host_set_scratch(PyObject *, PyObject *args) {
  int dev;
  unsigned long long stream, ptr, bytes;
  if (!PyArg_ParseTuple(args, "iKKK", &dev, &stream, &ptr, &bytes)) return nullptr;
  g_scratch[{dev, (void *)(uintptr_t)stream}] = Scratch{(void *)(uintptr_t)ptr, (size_t)bytes};
  Py_RETURN_NONE;
}

// bind({name: address}): the library's entry points
PyObject *host_bind(PyObject *, PyObject *args) {
  PyObject *d;
  if (!PyArg_ParseTuple(args, "O!", &PyDict_Type, &d)) return nullptr;
  const auto take = [&](const char *name, auto &slot) {
    PyObject *o = PyDict_GetItemString(d, name);
    void *p = o ? PyLong_AsVoidPtr(o) : nullptr;
    if (!p) {
      if (!PyErr_Occurred()) PyErr_Format(PyExc_KeyError, "%s", name);
      return false;
    }
    slot = (std::decay_t<decltype(slot)>)p;
    return true;
  };
  if (!take("wave_mxfp4_gemm", g_entry.gemm) || !take("wave_mxfp4_workspace_bytes", g_entry.workspace_bytes) ||
      !take("wave_mxfp4_gemm_grouped", g_entry.grouped) ||
      !take("wave_mxfp4_grouped_workspace_bytes", g_entry.grouped_workspace_bytes) ||
      !take("wave_mxfp4_gemm_gated_quantize", g_entry.gated) || !take("wave_mxfp8_gemm", g_entry.mxfp8) ||
      !take("wave_mxfp8_gemm_b_preshuffled", g_entry.mxfp8_b) ||
      !take("wave_mxfp8_workspace_bytes", g_entry.mxfp8_workspace_bytes) || !take("wave_mxfp4_quantize", g_entry.quantize) ||
      !take("wave_mxfp4_quantize_rows", g_entry.quantize_rows) ||
      !take("wave_mxfp4_moe_align_block_size", g_entry.moe_align) ||
      !take("wave_mxfp4_silu_and_mul_quantize", g_entry.silu_quantize))
    return nullptr;
  Py_RETURN_NONE;
}

#define WAVE_FAST(name) (PyCFunction)(void (*)(void))host_##name, METH_FASTCALL, nullptr
PyMethodDef g_methods[] = {{"bind", host_bind, METH_VARARGS, nullptr},
                           {"set_scratch", host_set_scratch, METH_VARARGS, nullptr},
                           {"gemm", WAVE_FAST(gemm)},
                           {"grouped", WAVE_FAST(grouped)},
                           {"gated", WAVE_FAST(gated)},
                           {"mxfp8", WAVE_FAST(mxfp8)},
                           {"quantize", WAVE_FAST(quantize)},
                           {"quantize_rows", WAVE_FAST(quantize_rows)},
                           {"moe_align", WAVE_FAST(moe_align)},
                           {"silu_quantize", WAVE_FAST(silu_quantize)},
                           {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_wave_host", "native call path of wave_amd", -1, g_methods};

}  // namespace

PyMODINIT_FUNC PyInit__wave_host(void) { return PyModule_Create(&g_module); }
