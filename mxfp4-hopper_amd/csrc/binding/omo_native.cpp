// _omo_native: the ordinary calls of the omo_python_api wrappers in one step
// of native code - checks, output allocation, launch and splits - for plain
// GPU tensors. A wrapper tries the function here first; None means that the
// call is not of the ordinary form (another type, layout, device or size, a
// tensor subclass, a torch mode or transform at work, an argument the entry
// point refuses), nothing was done, and the wrapper's Python code handles it,
// errors included. So each function accepts only what that code accepts and
// returns what it returns.
//
// Host time of a call (enqueued, not waited for) in Python and here: quantize
// of 16 x 7168 11.3 us and 4.4; dequant 11.8 and 3.6; FP8 requant in 8 splits
// 22.1 and 9.4, most of it the 16 views; 16 expert weights, 64 outputs, 176
// and 68.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <limits>
#include <vector>

#include "../../../include/omo_mxfp4.h"

namespace {

using at::Tensor;
using c10::DispatchKey;

constexpr auto kFp8 = at::kFloat8_e4m3fn;
constexpr float kEps = 1e-10f;  // of every wrapper without an eps argument

// Keys of tensors and threads whose operations mean more than their data:
// subclasses and modes in Python, functorch transforms, functionalization,
// lazy conjugation, negation and zeros.
const c10::DispatchKeySet kUnusual({DispatchKey::Python, DispatchKey::PythonTLSSnapshot, DispatchKey::FuncTorchBatched,
                                    DispatchKey::FuncTorchGradWrapper, DispatchKey::FuncTorchDynamicLayerFrontMode,
                                    DispatchKey::FuncTorchDynamicLayerBackMode, DispatchKey::FuncTorchVmapMode,
                                    DispatchKey::VmapMode, DispatchKey::Batched, DispatchKey::BatchedNestedTensor,
                                    DispatchKey::Functionalize, DispatchKey::Fake, DispatchKey::DeferredInit,
                                    DispatchKey::Conjugate, DispatchKey::Negative, DispatchKey::ZeroTensor});

// No torch mode or transform is at work on this thread.
bool quiet() {
  return !c10::impl::TorchDispatchModeTLS::any_modes_set() && at::impl::PythonTorchFunctionTLS::stack_len() == 0 &&
         !c10::impl::tls_local_dispatch_key_set().included_.has_any(kUnusual);
}

// The tensor behind o if it is a plain strided GPU tensor of this dtype, else
// an undefined one. Held by value: what runs without the GIL keeps its inputs
// whatever other threads do to o.
Tensor plain(PyObject* o, at::ScalarType dtype) {
  if (!THPVariable_CheckExact(o)) return {};
  const Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || t.scalar_type() != dtype ||
      t.key_set().has_any(kUnusual))
    return {};
  return t;
}

Tensor plain_matrix(PyObject* o, at::ScalarType dtype) {
  Tensor t = plain(o, dtype);
  if (t.defined() && (t.dim() != 2 || t.size(0) == 0 || t.size(1) == 0 || !t.is_contiguous())) t.reset();
  return t;
}

bool aligned(const Tensor& t, uintptr_t a) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & (a - 1)) == 0; }

Tensor empty_like_device(const Tensor& t, c10::IntArrayRef sizes, at::ScalarType dtype) {
  return at::empty(sizes, at::TensorOptions().device(t.device()).dtype(dtype));
}

hipStream_t stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// Raises the Python error of a C-ABI status, as omo's own check does.
bool ok(int status) {
  if (status == OMO_OK) return true;
  PyErr_SetString(status == OMO_ERR_UNSUPPORTED ? PyExc_NotImplementedError : PyExc_RuntimeError, omo_hip_last_error());
  return false;
}

PyObject* none() { Py_RETURN_NONE; }

// f() with the GIL released: allocation may free cached memory and wait for
// the device, and a launch waits while its queue is full; other threads of the
// program run meanwhile, as they do under torch.empty and ctypes. f calls no
// Python. Releasing and taking it back adds at most 0.1 us to a call (quantize
// of 16 x 7168, enqueued: 4.9 us before, 5.0 after).
template <typename F>
auto unlocked(F&& f) {
  struct Released {
    PyThreadState* state = PyEval_SaveThread();
    ~Released() { PyEval_RestoreThread(state); }
  } released;
  return f();
}

// A new tuple or list of tensors (steals nothing).
PyObject* tuple_of(const std::vector<Tensor>& ts) {
  PyObject* r = PyTuple_New((Py_ssize_t)ts.size());
  if (!r) return nullptr;
  for (size_t i = 0; i < ts.size(); i++) {
    PyObject* t = THPVariable_Wrap(ts[i]);
    if (!t) {
      Py_DECREF(r);
      return nullptr;
    }
    PyTuple_SET_ITEM(r, (Py_ssize_t)i, t);
  }
  return r;
}

PyObject* list_of(const std::vector<Tensor>& ts) {
  PyObject* r = PyList_New((Py_ssize_t)ts.size());
  if (!r) return nullptr;
  for (size_t i = 0; i < ts.size(); i++) {
    PyObject* t = THPVariable_Wrap(ts[i]);
    if (!t) {
      Py_DECREF(r);
      return nullptr;
    }
    PyList_SET_ITEM(r, (Py_ssize_t)i, t);
  }
  return r;
}

// (a, b), taking both references; null if either is.
PyObject* pair_of(PyObject* a, PyObject* b) {
  PyObject* r = a && b ? PyTuple_New(2) : nullptr;
  if (!r) {
    Py_XDECREF(a);
    Py_XDECREF(b);
    return nullptr;
  }
  PyTuple_SET_ITEM(r, 0, a);
  PyTuple_SET_ITEM(r, 1, b);
  return r;
}

// eps as a finite float, from a Python float only.
bool eps_of(PyObject* o, float* eps) {
  if (!PyFloat_CheckExact(o)) return false;
  const double d = PyFloat_AS_DOUBLE(o);
  if (!(d >= -std::numeric_limits<float>::max() && d <= std::numeric_limits<float>::max())) return false;
  *eps = (float)d;
  return true;
}

// Split lengths from a list or tuple of Python ints, none negative, summing
// to total; their count and sum of 128-row tiles.
bool splits_of(PyObject* o, int64_t total, std::vector<int64_t>* lens) {
  const bool list = PyList_CheckExact(o);
  if (!list && !PyTuple_CheckExact(o)) return false;
  const Py_ssize_t n = list ? PyList_GET_SIZE(o) : PyTuple_GET_SIZE(o);
  lens->resize((size_t)n);
  int64_t sum = 0;
  for (Py_ssize_t i = 0; i < n; i++) {
    PyObject* v = list ? PyList_GET_ITEM(o, i) : PyTuple_GET_ITEM(o, i);
    if (!PyLong_CheckExact(v)) return false;
    int over = 0;
    const long long m = PyLong_AsLongLongAndOverflow(v, &over);
    if (over || m < 0 || m > total - sum) return false;
    (*lens)[(size_t)i] = m;
    sum += m;
  }
  return sum == total;
}

bool arguments(const char* name, Py_ssize_t got, Py_ssize_t want) {
  if (got == want) return true;
  PyErr_Format(PyExc_TypeError, "%s takes %zd arguments, got %zd", name, want, got);
  return false;
}

// ------------------------------------------------------------------ quantize
// omo_per_token_group_quant_mxfp4(x)
PyObject* quantize(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (!arguments("quantize", n, 1)) return nullptr;
  const Tensor x = plain_matrix(a[0], at::kBFloat16);
  if (!x.defined() || x.size(1) % 32 != 0 || !aligned(x, 16) || !quiet()) return none();
  const int64_t M = x.size(0), K = x.size(1);
  const c10::DeviceGuard guard(x.device());
  Tensor q, s;
  if (!ok(unlocked([&] {
        q = empty_like_device(x, {M, K / 2}, at::kByte);
        s = empty_like_device(x, {M, K / 32}, at::kByte);
        return omo_hip_per_token_group_quant_fp4(x.data_ptr(), M * K, q.data_ptr(), M * K / 2, s.data_ptr(), M * K / 32,
                                                 32, kEps, -6.0f, 6.0f, 0, stream_of(x));
      })))
    return nullptr;
  return pair_of(THPVariable_Wrap(std::move(q)), THPVariable_Wrap(std::move(s)));
  END_HANDLE_TH_ERRORS
}

bool dual_takes(const Tensor& x) {
  return x.defined() && x.size(0) % 32 == 0 && x.size(1) % 32 == 0 && aligned(x, 16);
}

std::vector<Tensor> dual_outputs(const Tensor& x, int64_t M, int64_t K) {
  std::vector<Tensor> o;
  o.reserve(4);
  o.push_back(empty_like_device(x, {M, K / 2}, at::kByte));
  o.push_back(empty_like_device(x, {M, K / 32}, at::kByte));
  o.push_back(empty_like_device(x, {K, M / 2}, at::kByte));
  o.push_back(empty_like_device(x, {K, M / 32}, at::kByte));
  return o;
}

// omo_per_token_group_quant_mxfp4_dual(x, eps)
PyObject* quantize_dual(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (!arguments("quantize_dual", n, 2)) return nullptr;
  float eps;
  const Tensor x = plain_matrix(a[0], at::kBFloat16);
  if (!dual_takes(x) || !eps_of(a[1], &eps) || !quiet()) return none();
  const int64_t M = x.size(0), K = x.size(1), N = M * K;
  const c10::DeviceGuard guard(x.device());
  std::vector<Tensor> o;
  if (!ok(unlocked([&] {
        o = dual_outputs(x, M, K);
        return omo_hip_quant_mxfp4_dual(x.data_ptr(), M, K, o[0].data_ptr(), N / 2, o[1].data_ptr(), N / 32,
                                        o[2].data_ptr(), N / 2, o[3].data_ptr(), N / 32, eps, stream_of(x));
      })))
    return nullptr;
  return tuple_of(o);
  END_HANDLE_TH_ERRORS
}

// omo_per_token_group_quant_mxfp4_dual_grouped(xs, eps), xs a list or tuple
PyObject* quantize_dual_grouped(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (!arguments("quantize_dual_grouped", n, 2)) return nullptr;
  const bool list = PyList_CheckExact(a[0]);
  float eps;
  if ((!list && !PyTuple_CheckExact(a[0])) || !eps_of(a[1], &eps) || !quiet()) return none();
  const Py_ssize_t count = list ? PyList_GET_SIZE(a[0]) : PyTuple_GET_SIZE(a[0]);
  if (count == 0) return none();
  std::vector<Tensor> xs;
  std::vector<omo_dual_item> items;
  xs.reserve((size_t)count);
  items.reserve((size_t)count);
  for (Py_ssize_t i = 0; i < count; i++) {
    Tensor x = plain_matrix(list ? PyList_GET_ITEM(a[0], i) : PyTuple_GET_ITEM(a[0], i), at::kBFloat16);
    if (!dual_takes(x) || (i > 0 && x.device() != xs[0].device())) return none();
    items.push_back({nullptr, x.size(0), x.size(1), nullptr, 0, nullptr, 0, nullptr, 0, nullptr, 0});
    xs.push_back(std::move(x));
  }
  const c10::DeviceGuard guard(xs[0].device());
  std::vector<std::vector<Tensor>> outs(xs.size());
  if (!ok(unlocked([&] {
        for (size_t i = 0; i < xs.size(); i++) {
          const int64_t M = items[i].rows, K = items[i].cols, N = M * K;
          const std::vector<Tensor>& o = outs[i] = dual_outputs(xs[i], M, K);
          items[i] = {xs[i].data_ptr(), M, K, o[0].data_ptr(), N / 2, o[1].data_ptr(), N / 32,
                      o[2].data_ptr(), N / 2, o[3].data_ptr(), N / 32};
        }
        return omo_hip_quant_mxfp4_dual_grouped(items.data(), (int64_t)items.size(), eps, stream_of(xs[0]));
      })))
    return nullptr;
  PyObject* r = PyList_New(count);
  if (!r) return nullptr;
  for (Py_ssize_t i = 0; i < count; i++) {
    PyObject* t = tuple_of(outs[(size_t)i]);
    if (!t) {
      Py_DECREF(r);
      return nullptr;
    }
    PyList_SET_ITEM(r, i, t);
  }
  return r;
  END_HANDLE_TH_ERRORS
}

// ------------------------------------------------------------------- dequant
// omo_per_token_mxfp4ToBf16_dequant_wrapper(x, x_in_s, dtype), dtype bf16, fp16 or fp32
PyObject* dequantize(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (!arguments("dequantize", n, 3)) return nullptr;
  const Tensor x = plain_matrix(a[0], at::kByte), s = plain(a[1], at::kByte);
  if (!x.defined() || !s.defined() || !THPDtype_Check(a[2])) return none();
  const at::ScalarType dtype = reinterpret_cast<THPDtype*>(a[2])->scalar_type;
  const int type = dtype == at::kBFloat16 ? OMO_BF16 : dtype == at::kHalf ? OMO_F16 : dtype == at::kFloat ? OMO_F32 : -1;
  const int64_t M = x.size(0), half = x.size(1), scales = s.numel();
  if (type < 0 || half % 32 != 0 || M * half % 128 != 0 || !s.is_contiguous() || scales < M * half / 16 ||
      s.device() != x.device() || !aligned(x, 4) || !quiet())
    return none();
  const c10::DeviceGuard guard(x.device());
  Tensor y;
  if (!ok(unlocked([&] {
        y = empty_like_device(x, {M, 2 * half}, dtype);
        return omo_hip_Mxfp4_dequant(x.data_ptr(), M * half, s.data_ptr(), scales, y.data_ptr(), 2 * M * half, type,
                                     stream_of(x));
      })))
    return nullptr;
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

// --------------------------------------------------------------- FP8 requant
PyObject* split_pair(const Tensor& q, const Tensor& s, const std::vector<int64_t>& lens) {
  return pair_of(tuple_of(at::split_with_sizes(q, lens, 0)), tuple_of(at::split_with_sizes(s, lens, 1)));
}

// omo_per_token_mxfp4ToFp8_wrapper(x, x_in_s, m_splits)
PyObject* requant(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (!arguments("requant", n, 3)) return nullptr;
  const Tensor x = plain_matrix(a[0], at::kByte), s = plain_matrix(a[1], at::kByte);
  if (!x.defined() || !s.defined() || x.device() != s.device()) return none();
  const int64_t M = x.size(0), half = x.size(1), groups = (half + 63) / 64;
  std::vector<int64_t> lens;
  if (half % 16 != 0 || s.size(0) != M || s.size(1) != half / 16 || M * groups % 2 != 0 || !aligned(x, 8) ||
      (half % 64 == 0 && !aligned(s, 4)) || !splits_of(a[2], M, &lens) || !quiet())
    return none();
  const c10::DeviceGuard guard(x.device());
  Tensor q, qs;
  if (!ok(unlocked([&] {
        q = empty_like_device(x, {M, groups * 128}, kFp8);
        qs = empty_like_device(x, {groups, M}, at::kFloat);
        return omo_hip_Mxfp4ToFp8_padded(x.data_ptr(), M, half, s.data_ptr(), M * (half / 16), q.data_ptr(),
                                         M * groups * 128, qs.data_ptr(), groups * M, stream_of(x));
      })))
    return nullptr;
  return split_pair(half % 64 == 0 ? q : q.narrow(1, 0, 2 * half), qs, lens);
  END_HANDLE_TH_ERRORS
}

// ----------------------------------------------------------------- row -> col
// omo_per_token_mxfp4RowToBf16ToFp8Col_wrapper(data, scale, eps)
PyObject* row_to_col(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (!arguments("row_to_col", n, 3)) return nullptr;
  float eps;
  const Tensor x = plain_matrix(a[0], at::kByte), s = plain_matrix(a[1], at::kByte);
  if (!x.defined() || !s.defined() || x.device() != s.device() || !eps_of(a[2], &eps)) return none();
  const int64_t M = x.size(0), N = 2 * x.size(1), blocks = (N + 31) / 32, tiles = (M + 127) / 128;
  if (s.size(0) != M || s.size(1) != blocks || !quiet()) return none();
  const c10::DeviceGuard guard(x.device());
  Tensor q, qs;
  if (!ok(unlocked([&] {
        q = empty_like_device(x, {N, M}, kFp8);
        qs = empty_like_device(x, {tiles, N}, at::kFloat);
        return omo_hip_per_token_Mxfp4RowToBf16ToFp8Col(x.data_ptr(), M, N / 2, s.data_ptr(), M, blocks, q.data_ptr(), N,
                                                        M, qs.data_ptr(), tiles, N, eps, stream_of(x));
      })))
    return nullptr;
  return pair_of(THPVariable_Wrap(std::move(q)), THPVariable_Wrap(std::move(qs)));
  END_HANDLE_TH_ERRORS
}

// omo_per_token_mxfp4RowToBf16ToFp8Col_msplit_wrapper(data, scale, m_splits, eps), up to 128 splits by value
PyObject* row_to_col_splits(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (!arguments("row_to_col_splits", n, 4)) return nullptr;
  float eps;
  const Tensor x = plain_matrix(a[0], at::kByte), s = plain(a[1], at::kByte);
  if (!x.defined() || !s.defined() || x.device() != s.device() || !s.is_contiguous() || !eps_of(a[3], &eps))
    return none();
  const int64_t M = x.size(0), N = 2 * x.size(1), scales = s.numel();
  std::vector<int64_t> lens;
  if (!splits_of(a[2], M, &lens) || lens.size() > 128 || N % 32 != 0 || M >= ((int64_t)1 << 31) || !aligned(x, 16) ||
      scales < M * (N / 32) || !quiet())
    return none();
  std::vector<int64_t> tiles(lens.size());
  int64_t rows = 0;
  for (size_t i = 0; i < lens.size(); i++) rows += tiles[i] = (lens[i] + 127) / 128;
  const c10::DeviceGuard guard(x.device());
  Tensor q, qs;
  const int status = unlocked([&] {
    q = empty_like_device(x, {M * N}, kFp8);
    qs = empty_like_device(x, {rows, N}, at::kFloat);
    return omo_hip_Mxfp4RowToBf16ToFp8Col_splits(x.data_ptr(), M, N / 2, s.data_ptr(), scales, q.data_ptr(), M * N,
                                                 qs.data_ptr(), rows * N, lens.data(), (int64_t)lens.size(), eps,
                                                 stream_of(x));
  });
  if (status == OMO_ERR_UNSUPPORTED) return none();  // past one launch: device metadata
  if (!ok(status)) return nullptr;
  std::vector<Tensor> blocks;
  blocks.reserve(lens.size());
  int64_t at = 0;
  for (const int64_t m : lens) {
    blocks.push_back(q.as_strided({N, m}, {m > 0 ? m : 1, 1}, at * N));
    at += m;
  }
  return pair_of(list_of(blocks), list_of(at::split_with_sizes(qs, tiles, 0)));
  END_HANDLE_TH_ERRORS
}

// -------------------------------------------------------------- payload rows
// fp4_quantize_packed(x, eps)
PyObject* quantize_packed(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (!arguments("quantize_packed", n, 2)) return nullptr;
  float eps;
  const Tensor x = plain_matrix(a[0], at::kBFloat16);
  if (!x.defined() || x.size(1) % 128 != 0 || !aligned(x, 16) || !eps_of(a[1], &eps) || !quiet()) return none();
  const int64_t T = x.size(0), H = x.size(1);
  const c10::DeviceGuard guard(x.device());
  Tensor out;
  if (!ok(unlocked([&] {
        out = empty_like_device(x, {T, H / 32 * 17}, at::kByte);
        return omo_hip_quant_mxfp4_packed(x.data_ptr(), T, H, out.data_ptr(), out.numel(), eps, stream_of(x));
      })))
    return nullptr;
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// packed_mxfp4ToFp8(packed, m_splits), m_splits a list, a tuple or None
PyObject* requant_packed(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (!arguments("requant_packed", n, 2)) return nullptr;
  const Tensor p = plain_matrix(a[0], at::kByte);
  if (!p.defined() || p.size(1) % (17 * 4) != 0 || !aligned(p, 4)) return none();
  const int64_t T = p.size(0), H = p.size(1) / 17 * 32;
  std::vector<int64_t> lens;
  if ((a[1] != Py_None && !splits_of(a[1], T, &lens)) || !quiet()) return none();
  const c10::DeviceGuard guard(p.device());
  Tensor q, s;
  if (!ok(unlocked([&] {
        q = empty_like_device(p, {T, H}, kFp8);
        s = empty_like_device(p, {H / 128, T}, at::kFloat);
        return omo_hip_packed_Mxfp4ToFp8(p.data_ptr(), T, H, q.data_ptr(), q.numel(), s.data_ptr(), s.numel(),
                                         stream_of(p));
      })))
    return nullptr;
  if (a[1] != Py_None) return split_pair(q, s, lens);
  return pair_of(THPVariable_Wrap(std::move(q)), THPVariable_Wrap(std::move(s)));
  END_HANDLE_TH_ERRORS
}

// --------------------------------------------------------------- permutation
struct RowMap {
  Tensor src, dest;            // src: the row order, `rows` entries at its head
  int64_t rows = 0;
  std::vector<int64_t> loads;
  // what the call ended with: a status of the C ABI, a HIP error, or (wanted
  // >= 0) fewer rows wanted than the `rows` routed
  int status = OMO_OK;
  hipError_t hip = hipSuccess;
  int64_t wanted = -1;
};

// Raises the Python error of a row map that ended with one.
bool ok(const RowMap& r) {
  if (r.hip != hipSuccess) {
    PyErr_Format(PyExc_RuntimeError, "omo_route_counts: %s", hipGetErrorString(r.hip));
    return false;
  }
  if (r.wanted >= 0) {
    PyErr_Format(PyExc_ValueError, "num_out_tokens=%lld is smaller than the %lld routed tokens", (long long)r.wanted,
                 (long long)r.rows);
    return false;
  }
  return ok(r.status);
}

// A point of a stream that the host waits for. Pinned memory that a kernel
// ahead of the point writes stays with its owner until the kernel is done:
// destroyed with the wait outstanding (an exception, an early return), it waits.
class HostWait {
 public:
  HostWait() { e_ = hipEventCreateWithFlags(&event_, hipEventDisableTiming); }
  HostWait(const HostWait&) = delete;
  HostWait& operator=(const HostWait&) = delete;
  ~HostWait() {
    if (pending_) (void)hipEventSynchronize(event_);
    if (event_) (void)hipEventDestroy(event_);
  }
  hipError_t created() const { return e_; }
  // Covers the work enqueued on the stream before the call.
  hipError_t record(hipStream_t stream) {
    const hipError_t e = hipEventRecord(event_, stream);
    if (e == hipSuccess) pending_ = true;
    else (void)hipStreamSynchronize(stream);
    return e;
  }
  hipError_t wait() {
    pending_ = false;
    return hipEventSynchronize(event_);
  }

 private:
  hipEvent_t event_ = nullptr;
  hipError_t e_;
  bool pending_ = false;
};

// num_out: rows asked for, or -1. `ahead`: the order is enqueued before the
// host waits for the loads, so that nothing is left to do after the wait; with
// num_out < 0 its length is not known then and src is scratch for every pair.
// Everything whose size is known is allocated before the first launch. Runs
// without the GIL.
RowMap row_map(const Tensor& map, int64_t T, int64_t E, int64_t num_out, bool want_dest, bool ahead) {
  RowMap r;
  const int64_t chunks = omo_hip_route_chunks(T, E);
  const hipStream_t stream = stream_of(map);
  const Tensor counts = empty_like_device(map, {E * chunks}, at::kInt);
  // The counts also go to pinned host memory, so that the host waits for the
  // counting launch alone and no copy follows it.
  const Tensor seen = at::empty({E * chunks}, at::TensorOptions().dtype(at::kInt).pinned_memory(true));
  if (want_dest) r.dest = empty_like_device(map, {T, E}, at::kInt);
  if (ahead) r.src = empty_like_device(map, {num_out < 0 ? T * E : num_out}, at::kInt);
  HostWait counted;
  if ((r.hip = counted.created()) != hipSuccess) return r;
  r.status = omo_hip_route_counts(map.data_ptr(), T, E, counts.data_ptr<int32_t>(), E * chunks,
                                  seen.data_ptr<int32_t>(), stream);
  if (r.status != OMO_OK || (r.hip = counted.record(stream)) != hipSuccess) return r;
  const auto order = [&](bool pad) {
    const int64_t rows = r.src.numel();
    r.status = omo_hip_route_rows(map.data_ptr(), T, E, counts.data_ptr<int32_t>(), E * chunks,
                                  rows ? r.src.data_ptr<int32_t>() : nullptr, rows, pad,
                                  want_dest ? r.dest.data_ptr<int32_t>() : nullptr, want_dest ? T * E : 0, stream);
  };
  if (ahead) order(num_out >= 0);
  if (r.status != OMO_OK || (r.hip = counted.wait()) != hipSuccess) return r;
  const int32_t* c = seen.data_ptr<int32_t>();
  int64_t routed = 0;
  r.loads.assign((size_t)E, 0);
  for (int64_t i = 0; i < E; i++) {
    for (int64_t k = 0; k < chunks; k++) r.loads[(size_t)i] += c[i * chunks + k];
    routed += r.loads[(size_t)i];
  }
  r.rows = num_out < 0 || num_out < routed ? routed : num_out;
  if (num_out >= 0 && num_out < routed) {
    r.wanted = num_out;
  } else if (!ahead) {
    r.src = empty_like_device(map, {r.rows}, at::kInt);
    order(num_out > routed);
  }
  return r;
}

// A routing map that the two row-map launches take and are the faster for. A
// workgroup covers four experts and one of at most 64 chunks of tokens: one or
// two experts of very many tokens leave the chip idle (row map and loads, us,
// against the torch composition: 2^22 x 1 289 and 269, 3 * 2^20 x 1 202 and
// 246, 2^23 x 2 641 and 620, 2^22 x 2 328 and 383; 2^24 x 4 1341 and 1565). And each
// sums the counts before its own, so the work grows with the square of experts
// times chunks (4096 x 65536 8691 and 2890, 4096 x 16384 959 and 881, 512 x
// 65536 848 and 786; 4096 x 8192 400 and 528).
Tensor plain_map(PyObject* o) {
  Tensor t = plain_matrix(o, at::kBool);
  if (!t.defined()) return t;
  const int64_t T = t.size(0), E = t.size(1);
  if (T >= ((int64_t)1 << 31) / E || E > 4 * 65534 || (E <= 2 && T >= E << 22) ||
      E * omo_hip_route_chunks(T, E) >= (int64_t)1 << 17)
    t.reset();
  return t;
}

// Raises where the map's stream is being captured: the host has to read the
// loads, and a counting launch recorded without that would write the pinned
// counts again on every replay, whoever holds them by then.
bool uncaptured(const Tensor& map) {
  hipStreamCaptureStatus s = hipStreamCaptureStatusNone;
  const hipError_t e = hipStreamIsCapturing(stream_of(map), &s);
  if (e == hipSuccess && s == hipStreamCaptureStatusNone) return true;
  PyErr_SetString(PyExc_RuntimeError,
                  "the host reads the expert loads of a routing map: not permitted while its stream is being captured");
  return false;
}

// None (-1) or a Python int in [0, 2^31).
bool num_out_of(PyObject* o, int64_t* num_out) {
  *num_out = -1;
  if (o == Py_None) return true;
  if (!PyLong_CheckExact(o)) return false;
  int over = 0;
  *num_out = PyLong_AsLongLongAndOverflow(o, &over);
  return !over && *num_out >= 0 && *num_out < ((int64_t)1 << 31);
}

PyObject* list_of_ints(const std::vector<int64_t>& v) {
  PyObject* r = PyList_New((Py_ssize_t)v.size());
  if (!r) return nullptr;
  for (size_t i = 0; i < v.size(); i++) {
    PyObject* x = PyLong_FromLongLong(v[i]);
    if (!x) {
      Py_DECREF(r);
      return nullptr;
    }
    PyList_SET_ITEM(r, (Py_ssize_t)i, x);
  }
  return r;
}

// make_row_id_map(routing_map, num_out_tokens) of a bool map -> (src, loads, dest)
PyObject* make_row_map(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (!arguments("make_row_map", n, 2)) return nullptr;
  int64_t num_out;
  const Tensor map = plain_map(a[0]);
  if (!map.defined() || !num_out_of(a[1], &num_out) || !quiet()) return none();
  const int64_t T = map.size(0), E = map.size(1);
  const c10::DeviceGuard guard(map.device());
  if (!uncaptured(map)) return nullptr;
  RowMap m = unlocked([&] { return row_map(map, T, E, num_out, true, false); });
  if (!ok(m)) return nullptr;
  PyObject* loads = list_of_ints(m.loads);
  PyObject* rest = pair_of(loads, THPVariable_Wrap(std::move(m.dest)));
  PyObject* head = rest ? THPVariable_Wrap(std::move(m.src)) : nullptr;
  PyObject* r = head ? PyTuple_Pack(3, head, PyTuple_GET_ITEM(rest, 0), PyTuple_GET_ITEM(rest, 1)) : nullptr;
  Py_XDECREF(head);
  Py_XDECREF(rest);
  return r;
  END_HANDLE_TH_ERRORS
}

// Rows of a code or scale matrix, perhaps strided: bytes from the first to past the last.
bool rows_of(const Tensor& t, int64_t* span, int64_t* stride) {
  if (t.dim() != 2 || t.size(0) == 0 || t.size(1) == 0 || (t.size(1) > 1 && t.stride(1) != 1)) return false;
  *stride = t.size(0) > 1 ? t.stride(0) : t.size(1);
  *span = (t.size(0) - 1) * *stride + t.size(1);
  return true;
}

// mxfp4_permute_to_fp8(codes, scales, routing_map, num_out_tokens) unsplit -> (fp8, scales, src, loads)
PyObject* permute_to_fp8(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (!arguments("permute_to_fp8", n, 4)) return nullptr;
  int64_t num_out, cspan, cstride, sspan, sstride;
  const Tensor codes = plain(a[0], at::kByte), scales = plain(a[1], at::kByte), map = plain_map(a[2]);
  if (!codes.defined() || !scales.defined() || !map.defined() || !num_out_of(a[3], &num_out) ||
      !rows_of(codes, &cspan, &cstride) || !rows_of(scales, &sspan, &sstride))
    return none();
  const int64_t T = codes.size(0), H = 2 * codes.size(1), map_T = map.size(0), E = map.size(1);
  if (scales.size(0) != T || H % 128 != 0 || scales.size(1) != H / 32 || cstride < H / 2 || sstride < H / 32 ||
      cstride % 4 != 0 || sstride % 4 != 0 || !aligned(codes, 4) || !aligned(scales, 4) ||
      codes.device() != map.device() || scales.device() != map.device() || !quiet())
    return none();
  const c10::DeviceGuard guard(map.device());
  if (!uncaptured(map)) return nullptr;
  RowMap m;
  Tensor src, q, s;
  const int status = unlocked([&]() -> int {
    // The order goes ahead of the wait; the requant, which has to know the
    // number of rows, copies it from the scratch to its own buffer.
    m = row_map(map, map_T, E, num_out, false, true);
    if (m.status != OMO_OK || m.hip != hipSuccess || m.wanted >= 0) return OMO_OK;  // raised below
    const int64_t N = m.rows;
    const bool scratch = m.src.numel() != N;
    src = scratch ? empty_like_device(codes, {N}, at::kInt) : m.src;
    q = empty_like_device(codes, {N, H}, kFp8);
    s = empty_like_device(codes, {H / 128, N}, at::kFloat);
    if (N == 0) return OMO_OK;
    return omo_hip_permute_Mxfp4ToFp8_copy(codes.data_ptr(), cspan, cstride, scales.data_ptr(), sspan, sstride, T, H,
                                           m.src.data_ptr<int32_t>(), N,
                                           scratch ? src.data_ptr<int32_t>() : nullptr, q.data_ptr(), q.numel(),
                                           s.data_ptr(), s.numel(), stream_of(codes));
  });
  if (!ok(m) || !ok(status)) return nullptr;
  PyObject* loads = list_of_ints(m.loads);
  PyObject* ts = loads ? tuple_of({q, s, src}) : nullptr;
  PyObject* r = ts ? PyTuple_Pack(4, PyTuple_GET_ITEM(ts, 0), PyTuple_GET_ITEM(ts, 1), PyTuple_GET_ITEM(ts, 2), loads)
                   : nullptr;
  Py_XDECREF(ts);
  Py_XDECREF(loads);
  return r;
  END_HANDLE_TH_ERRORS
}

#define METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {METHOD(quantize),       METHOD(quantize_dual),     METHOD(quantize_dual_grouped),
                          METHOD(dequantize),     METHOD(requant),           METHOD(row_to_col),
                          METHOD(row_to_col_splits), METHOD(quantize_packed), METHOD(requant_packed),
                          METHOD(make_row_map),   METHOD(permute_to_fp8),    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_omo_native", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__omo_native() {
  PyObject* m = PyModule_Create(&kModule);
  if (m && PyModule_AddStringConstant(m, "torch_version", OMO_TORCH_VERSION) != 0) Py_CLEAR(m);
  return m;
}
