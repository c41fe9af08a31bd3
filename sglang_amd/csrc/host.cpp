// The layer-level entry points of sglang_amd as one native call each.
//
// What bounds a decode step here is not the GPU: a block-FP8 linear at M = 1 is 13 us of kernels, and its pass through
// Python (argument checks, two dispatcher calls into Python implementations, four allocations, ctypes with twenty arguments)
// took 38 us; the fused expert layer took 130 us.  A function of this module checks the operands, takes all its scratch from
// torch's caching allocator in one piece and makes the C ABI calls back to back: 5 to 8 us for a linear.
//
// Every function returns None, before anything has been launched, for operands that it does not take as they are: tensors of
// a mode or a subclass (of the dispatcher's - tracing, fake tensors - or with a __torch_function__), inputs that want gradients, unusual types and layouts, and everything
// that is an error.  The Python caller then goes through the dispatcher ops, which know all cases and word the errors.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/grad_mode.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/record_function.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Device.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <initializer_list>
#include <map>
#include <mutex>
#include <vector>

#include "../../include/fp8k.h"

namespace {

using at::Tensor;
using c10::DispatchKey;
using c10::DispatchKeySet;
using c10::ScalarType;

constexpr float kEps = 1e-10f;

PyObject* g_has_torch_function = nullptr;  // torch.overrides.has_torch_function_unary
PyObject* g_workspaces = nullptr;     // sgl_kernel._workspaces: (device index, stream) -> the buffer of that stream
PyObject* g_grow_workspace = nullptr; // sgl_kernel._workspace

// ---------------------------------------------------------------------------------------------- operands
// A mode is active that has to see the ops: a torch function mode, or one of the dispatcher (tracing, fake tensors,
// functionalisation, vmap).
bool modes_active() {
  if (at::impl::torch_function_mode_enabled()) return true;
  constexpr DispatchKeySet modes({DispatchKey::Python, DispatchKey::PythonTLSSnapshot, DispatchKey::Functionalize,
                                  DispatchKey::FuncTorchDynamicLayerFrontMode, DispatchKey::FuncTorchBatched,
                                  DispatchKey::Tracer});
  return c10::impl::tls_local_dispatch_key_set().included_.has_any(modes);
}

// A strided GPU tensor with nothing between it and its memory, on the device of the call.
bool plain(const Tensor& t, int device) {
  constexpr DispatchKeySet odd({DispatchKey::Python, DispatchKey::PythonTLSSnapshot, DispatchKey::Functionalize,
                                DispatchKey::FuncTorchBatched, DispatchKey::FuncTorchGradWrapper, DispatchKey::Conjugate,
                                DispatchKey::Negative, DispatchKey::ZeroTensor});
  if (!t.defined() || t.key_set().has_any(odd) || t.is_nested()) return false;
  if (!t.is_cuda() || t.layout() != c10::kStrided || t.get_device() != device) return false;
  return !(t.requires_grad() && at::GradMode::is_enabled());
}

// a tensor whose class has no say in what is done with it: a subclass may have a __torch_function__ without being a dispatcher
// subclass; parameters and subclasses that switch theirs off have none
bool tensor_arg(PyObject* o, Tensor& t) {
  if (!THPVariable_CheckExact(o)) {  // neither a Tensor nor a Parameter
    if (!THPVariable_Check(o)) return false;
    PyObject* const has = PyObject_CallFunctionObjArgs(g_has_torch_function, o, nullptr);
    if (!has) throw python_error();
    Py_DECREF(has);  // True or False
    if (has != Py_False) return false;
  }
  t = THPVariable_Unpack(o);
  return true;
}

bool truth(PyObject* o) {
  if (o == Py_True || o == Py_False) return o == Py_True;
  const int is = PyObject_IsTrue(o);
  if (is < 0) throw python_error();
  return is == 1;
}

bool is_fp8(const Tensor& t) { return t.scalar_type() == ScalarType::Float8_e4m3fn; }
bool is_half(ScalarType t) { return t == ScalarType::BFloat16 || t == ScalarType::Half; }

int code(ScalarType t) {
  return t == ScalarType::BFloat16 ? FP8K_BF16 : t == ScalarType::Half ? FP8K_F16 : FP8K_F32;
}

bool non_negative_strides(const Tensor& t) {
  for (int64_t s : t.strides())
    if (s < 0) return false;
  return true;
}

bool is_128x128(PyObject* o) {
  if (!PyList_Check(o) && !PyTuple_Check(o)) return false;
  if (PySequence_Fast_GET_SIZE(o) != 2) return false;
  for (int i = 0; i < 2; ++i) {
    PyObject* v = PySequence_Fast_GET_ITEM(o, i);
    if (!PyLong_CheckExact(v) || PyLong_AsLong(v) != 128) return false;
  }
  return true;
}

int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }
int64_t ceil_to(int64_t a, int64_t b) { return ceil_div(a, b) * b; }

// a weight with its 128 x 128 block scales: w e4m3fn [N, K] contiguous, scale float32 [ceil(N/128), ceil(K/128)]
bool block_weight(const Tensor& w, const Tensor& s, int64_t K, int device) {
  if (!plain(w, device) || !plain(s, device) || !is_fp8(w) || w.dim() != 2 || w.size(1) != K || !w.is_contiguous()) return false;
  if (s.scalar_type() != ScalarType::Float || s.dim() != 2 || !non_negative_strides(s)) return false;
  const int64_t N = w.size(0);
  return N > 0 && N % 8 == 0 && s.size(0) == ceil_div(N, 128) && s.size(1) == ceil_div(K, 128);
}

void check(int status) {
  if (status != 0) {
    const char* msg = fp8k_last_error();
    throw std::runtime_error(msg && *msg ? msg : "fp8k error");
  }
}

// ---------------------------------------------------------------------------------------------- memory
Tensor empty(at::IntArrayRef size, ScalarType t, const at::Device& d) {
  return Tensor(at::detail::empty_cuda(size, t, d, std::nullopt));
}

// [rows, cols] with strides (1, ld): column-major, every column padded to ld entries
Tensor empty_column_major(int64_t rows, int64_t cols, int64_t ld, ScalarType t, const at::Device& d) {
  Tensor out = empty({cols * ld}, t, d);
  out.unsafeGetTensorImpl()->set_sizes_and_strides(at::IntArrayRef({rows, cols}), at::IntArrayRef({(int64_t)1, ld}));
  return out;
}

// The scratch of one call: one block of torch's caching allocator on the call's stream, cut into 256-byte aligned pieces.  It
// goes back when the call returns; the allocator hands it out again on the same stream only (or, under graph capture, inside
// the capture's pool), so launches that are still queued keep it to themselves, whatever other threads and streams do.
class Scratch {
 public:
  Scratch(size_t bytes, hipStream_t st) {
    if (bytes) base_ = static_cast<char*>(c10::hip::HIPCachingAllocator::raw_alloc_with_stream(bytes, st));
  }
  ~Scratch() {
    if (base_) c10::hip::HIPCachingAllocator::raw_delete(base_);
  }
  Scratch(const Scratch&) = delete;
  Scratch& operator=(const Scratch&) = delete;
  static size_t room(int64_t bytes) { return (size_t)ceil_to(bytes, 256); }
  template <class T = void>
  T* take(int64_t bytes) {
    char* p = base_ + used_;
    used_ += room(bytes);
    return reinterpret_cast<T*>(p);
  }

 private:
  char* base_ = nullptr;
  size_t used_ = 0;
};

// What allocates or launches runs without the interpreter lock: a launch into a full queue and an allocation that has to free
// cached blocks wait for the device, and other Python threads, one of which the device may be waiting for, must not wait with it.
class WithoutGil {
 public:
  WithoutGil() : state_(PyEval_SaveThread()) {}
  ~WithoutGil() { PyEval_RestoreThread(state_); }
  WithoutGil(const WithoutGil&) = delete;
  WithoutGil& operator=(const WithoutGil&) = delete;

 private:
  PyThreadState* state_;
};

// the part of a call that works on the device: no interpreter lock, the call's device made current, and its stream
struct Call {
  explicit Call(const Tensor& t)
      : guard(t.device()), device(t.get_device()), stream(c10::hip::getCurrentHIPStream(t.get_device()).stream()) {}
  WithoutGil unlocked;  // first: taken back last
  c10::DeviceGuard guard;
  int device;
  hipStream_t stream;
};

// the GEMM workspace of the current stream (sgl_kernel._workspace): nullptr and false when the Python side raised.  Asked for
// with the interpreter lock; what it returns is never released.
bool stream_workspace(const Tensor& like, int64_t need, void*& p, int64_t& bytes) {
  p = nullptr;
  bytes = 0;
  if (need <= 0) return true;
  const hipStream_t st = c10::hip::getCurrentHIPStream(like.get_device()).stream();
  PyObject* key = Py_BuildValue("(iK)", (int)like.get_device(), (unsigned long long)(uintptr_t)st);
  if (!key) return false;
  PyObject* buf = PyDict_GetItem(g_workspaces, key);  // borrowed
  Py_DECREF(key);
  if (buf && THPVariable_Check(buf)) {
    const Tensor& t = THPVariable_Unpack(buf);
    if (t.numel() >= need) {
      p = t.data_ptr();
      bytes = t.numel();
      return true;
    }
  }
  PyObject* device = THPDevice_New(like.device());
  PyObject* got = device ? PyObject_CallFunction(g_grow_workspace, "OL", device, (long long)need) : nullptr;
  Py_XDECREF(device);
  if (!got) return false;
  const Tensor& t = THPVariable_Unpack(got);
  p = t.data_ptr();
  bytes = t.numel();
  Py_DECREF(got);  // the registry keeps it
  return true;
}

// Threads that share a stream share its workspace: the launches of one product (copy of the scales, GEMM, reduction) go onto the
// stream together.  One lock per workspace, so a thread waits for launches onto its own stream only; taken without the interpreter lock.
std::mutex& workspace_lock(const void* workspace) {
  static std::mutex mutex;
  static auto* const locks = new std::map<const void*, std::mutex>;  // as many as there are workspaces; both live as long as the process
  std::lock_guard<std::mutex> lock(mutex);
  return (*locks)[workspace];
}

// A record of the call for torch's profiler and other observers, as the dispatcher keeps one of an op: for the rest of the scope.
#define OBSERVED(name, ...) RECORD_FUNCTION("fp8k::" name, (std::vector<c10::IValue>{__VA_ARGS__}))

// an argument that did not convert is the dispatcher path's to word as well
#define DECLINE     \
  do {              \
    PyErr_Clear();  \
    Py_RETURN_NONE; \
  } while (0)

// ---------------------------------------------------------------------------------------------- group quant
// group_quant(x, group_size, eps, column_major, tma_aligned, ue8m0, fuse_silu) -> (q, scales) or None
PyObject* group_quant(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor x;
  if (n != 7 || !tensor_arg(a[0], x) || modes_active() || !x.is_cuda() || !plain(x, x.get_device())) DECLINE;
  if (!PyLong_Check(a[1]) || !PyFloat_Check(a[2])) DECLINE;
  const int64_t group = PyLong_AsLongLong(a[1]);
  const float eps = (float)PyFloat_AS_DOUBLE(a[2]);
  const bool column = truth(a[3]), tma = truth(a[4]), ue8m0 = truth(a[5]), fuse = truth(a[6]);
  const ScalarType dt = x.scalar_type();
  if (!(is_half(dt) || dt == ScalarType::Float) || x.dim() < 1 || x.numel() == 0 || !x.is_contiguous()) DECLINE;
  if ((column || ue8m0) && x.dim() != 2) DECLINE;
  if (ue8m0 && !(column && tma && group == 128)) DECLINE;
  const int64_t width = x.size(-1);
  const int64_t K = fuse ? width / 2 : width;
  if (group <= 0 || width % group != 0 || K % group != 0 || K == 0 || (fuse && (width % 2 != 0 || group != 128))) DECLINE;
  const int64_t M = x.numel() / width, G = K / group;

  Tensor q, s;
  {
    Call c(x);
    OBSERVED("group_quant", x);
    c10::SmallVector<int64_t, 5> shape(x.sizes().begin(), x.sizes().end());
    shape.back() = K;
    q = empty(shape, ScalarType::Float8_e4m3fn, x.device());
    int64_t sm, sg;
    if (ue8m0) {
      sm = 1;
      sg = ceil_to(M, 4);
      s = empty_column_major(M, ceil_div(G, 4), sg, ScalarType::Int, x.device());
    } else if (column) {
      sm = 1;
      sg = tma ? ceil_to(M, 4) : M;
      s = empty_column_major(M, G, sg, ScalarType::Float, x.device());
    } else {
      shape.back() = G;
      s = empty(shape, ScalarType::Float, x.device());
      sm = G;
      sg = 1;
    }
    check((fuse ? fp8k_silu_mul_group_quant : fp8k_group_quant)(
        x.data_ptr(), q.data_ptr(), s.data_ptr(), M, K, group, eps, -448.f, 448.f, code(dt), sm, sg,
        ue8m0 ? FP8K_SCALE_UE8M0_PACKED : FP8K_SCALE_F32, c.stream));
  }
  PyObject* out = PyTuple_New(2);
  if (!out) return nullptr;
  PyTuple_SET_ITEM(out, 0, THPVariable_Wrap(std::move(q)));
  PyTuple_SET_ITEM(out, 1, THPVariable_Wrap(std::move(s)));
  return out;
  END_HANDLE_TH_ERRORS
}

// ---------------------------------------------------------------------------------------------- block-FP8 GEMM
// block_linear(x, weight, block_size, weight_scale, bias) -> output or None: group quant, GEMM, bias
PyObject* block_linear(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor x, w, ws, bias;
  if (n != 5 || modes_active() || !tensor_arg(a[0], x) || !tensor_arg(a[1], w) || !is_128x128(a[2]) || !tensor_arg(a[3], ws)) DECLINE;
  if (!x.is_cuda()) DECLINE;
  const int dev = x.get_device();
  const ScalarType dt = x.scalar_type();
  if (!plain(x, dev) || !is_half(dt) || x.dim() < 1 || x.numel() == 0 || !x.is_contiguous()) DECLINE;
  const int64_t K = x.size(-1), M = x.numel() / K;
  if (K % 128 != 0 || !block_weight(w, ws, K, dev)) DECLINE;
  const int64_t N = w.size(0);
  if (a[4] != Py_None) {
    if (!tensor_arg(a[4], bias) || !plain(bias, dev) || bias.dim() != 1 || bias.size(0) != N || bias.scalar_type() != dt || !bias.is_contiguous()) DECLINE;
  }

  Tensor out;
  {
    Call c(x);
    OBSERVED("block_linear", x, w, ws, bias);
    c10::SmallVector<int64_t, 5> shape(x.sizes().begin(), x.sizes().end());
    shape.back() = N;
    out = empty(shape, dt, x.device());
    const int64_t wsb = fp8k_linear_workspace_bytes(M, N, K, 1);
    Scratch mem(wsb, c.stream);
    check(fp8k_block_linear(x.data_ptr(), w.data_ptr(), ws.data_ptr<float>(), bias.defined() ? bias.data_ptr() : nullptr, out.data_ptr(), M,
                            N, K, K, ws.stride(0), ws.stride(1), N, kEps, code(dt), wsb ? mem.take(wsb) : nullptr, wsb, c.stream));
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// block_matmul(A, B, As, Bs, block_size, out_dtype, scales_pow2) -> C or None: the GEMM on quantised activations, with
// float32 activation scales or, where the weight scales are known to be powers of two, packed UE8M0 ones
PyObject* block_matmul(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor x, w, xs, ws;
  if (n != 7 || modes_active() || !tensor_arg(a[0], x) || !tensor_arg(a[1], w) || !tensor_arg(a[2], xs) || !tensor_arg(a[3], ws))
    DECLINE;
  if (!is_128x128(a[4]) || !THPDtype_Check(a[5]) || !x.is_cuda()) DECLINE;
  const int dev = x.get_device();
  const ScalarType dt = reinterpret_cast<THPDtype*>(a[5])->scalar_type;
  const bool pow2 = truth(a[6]);
  if (!plain(x, dev) || !is_fp8(x) || x.dim() != 2 || x.numel() == 0 || !x.is_contiguous() || !is_half(dt)) DECLINE;
  const int64_t M = x.size(0), K = x.size(1), kb = ceil_div(K, 128);
  if (K % 16 != 0 || !block_weight(w, ws, K, dev)) DECLINE;
  const int64_t N = w.size(0);
  if (!plain(xs, dev) || xs.dim() != 2 || xs.size(0) != M || !non_negative_strides(xs)) DECLINE;
  const bool packed = xs.scalar_type() == ScalarType::Int;
  if (packed) {
    // the matrix core applies the exponents in the tile kernels only (above 128 rows)
    if (!pow2 || M <= 128 || K % 128 != 0 || xs.size(1) != ceil_div(kb, 4)) DECLINE;
  } else if (xs.scalar_type() != ScalarType::Float || xs.size(1) != kb) {
    DECLINE;
  }

  void* work;
  int64_t bytes;
  if (!stream_workspace(x, fp8k_block_gemm_workspace_bytes(M, N, K), work, bytes)) return nullptr;
  Tensor out;
  {
    Call c(x);
    OBSERVED("block_matmul", x, w, xs, ws);
    out = empty({M, N}, dt, x.device());
    std::unique_lock<std::mutex> together;
    if (work) together = std::unique_lock<std::mutex>(workspace_lock(work));
    if (packed)
      check(fp8k_block_gemm_ue8m0(x.data_ptr(), w.data_ptr(), xs.data_ptr<int32_t>(), ws.data_ptr<float>(), out.data_ptr(), M, N, K, K,
                                  K, xs.stride(0), xs.stride(1), ws.stride(0), ws.stride(1), N, code(dt), work, bytes, c.stream));
    else
      check(fp8k_block_gemm(x.data_ptr(), w.data_ptr(), xs.data_ptr<float>(), ws.data_ptr<float>(), out.data_ptr(), M, N, K, K, K,
                            xs.stride(0), xs.stride(1), ws.stride(0), ws.stride(1), N, code(dt), work, bytes, c.stream));
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// ---------------------------------------------------------------------------------------------- per-token linear
// token_linear(x, weight, weight_scale, bias, per_token) -> output or None: dynamic per-token quant, row-scaled GEMM, bias.
// per_token: the caller asked for per-token scales; without it only a per-channel weight scale implies them.
PyObject* token_linear(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor x, w, ws, bias;
  if (n != 5 || modes_active() || !tensor_arg(a[0], x) || !tensor_arg(a[1], w) || !tensor_arg(a[2], ws) || !x.is_cuda()) DECLINE;
  const int dev = x.get_device();
  const ScalarType dt = x.scalar_type();
  if (!plain(x, dev) || !is_half(dt) || x.dim() < 1 || x.numel() == 0 || !x.is_contiguous()) DECLINE;
  const int64_t K = x.size(-1), M = x.numel() / K;
  if (!plain(w, dev) || !is_fp8(w) || w.dim() != 2 || w.size(0) != K || K % 16 != 0 || K <= 1) DECLINE;
  const int64_t N = w.size(1);
  if (N <= 0 || N % 8 != 0 || w.stride(0) != 1 || (N > 1 && w.stride(1) < K)) DECLINE;
  if (!plain(ws, dev) || ws.scalar_type() != ScalarType::Float || !ws.is_contiguous()) DECLINE;
  if (ws.numel() != N && !(ws.numel() == 1 && truth(a[4]))) DECLINE;
  if (a[3] != Py_None) {
    if (!tensor_arg(a[3], bias) || !plain(bias, dev) || bias.numel() != N || !bias.is_contiguous()) DECLINE;
    if (bias.scalar_type() != dt && bias.scalar_type() != ScalarType::Float) DECLINE;
  }

  Tensor out;
  {
    Call c(x);
    OBSERVED("token_linear", x, w, ws, bias);
    c10::SmallVector<int64_t, 5> shape(x.sizes().begin(), x.sizes().end());
    shape.back() = N;
    out = empty(shape, dt, x.device());
    const int64_t wsb = fp8k_linear_workspace_bytes(M, N, K, 0);
    Scratch mem(wsb, c.stream);
    check(fp8k_token_linear(x.data_ptr(), w.data_ptr(), ws.data_ptr<float>(), ws.numel() == 1 ? 0 : 1, bias.defined() ? bias.data_ptr() : nullptr,
                            bias.defined() ? code(bias.scalar_type()) : FP8K_F32, out.data_ptr(), M, N, K, N > 1 ? w.stride(1) : K, N, code(dt),
                            wsb ? mem.take(wsb) : nullptr, wsb, c.stream));
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// ---------------------------------------------------------------------------------------------- absorbed products
// Three zeroed int32 per (device, stream) for fp8k_tensor_quant_mla_sync, made on first use and kept: at most kMaxSync of them.  What
// makes one stream of a handle are torch's own streams, which live as long as the process.  A stream that came in from outside (its
// id is its handle) may be destroyed and its handle given to another while launches are queued, and hipStreamPerThread is one handle
// for a stream of every thread.  Those get none and take the two launches, as do calls under graph capture, whose replays may
// run on any stream.
constexpr size_t kMaxSync = 64;
int32_t* stream_sync(const Tensor& like, const c10::hip::HIPStream& stream) {
  const hipStream_t st = stream.stream();
  if (st && (uint64_t)stream.id() == (uint64_t)(uintptr_t)st) return nullptr;
  hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(st, &capturing) != hipSuccess) {
    (void)hipGetLastError();  // the launches report what is wrong with the stream, not this question
    return nullptr;
  }
  if (capturing != hipStreamCaptureStatusNone) return nullptr;
  static std::mutex mutex;
  static auto* const words = new std::map<std::pair<int, hipStream_t>, Tensor>;  // lives as long as the process
  const auto key = std::make_pair((int)like.get_device(), st);
  {
    std::lock_guard<std::mutex> lock(mutex);
    const auto it = words->find(key);
    if (it != words->end()) return it->second.data_ptr<int32_t>();
    if (words->size() >= kMaxSync) return nullptr;
  }
  // outside the lock, as it may wait for the device; of two threads on one stream the first to come back decides
  Tensor fresh = at::zeros({3}, like.options().dtype(ScalarType::Int));  // on the current stream, which is st
  std::lock_guard<std::mutex> lock(mutex);
  return words->emplace(key, std::move(fresh)).first->second.data_ptr<int32_t>();
}

// mla_quant(x, x_s, eps) -> x_q or None
PyObject* mla_quant(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor x, s;
  if (n != 3 || modes_active() || !tensor_arg(a[0], x) || !tensor_arg(a[1], s) || !PyFloat_Check(a[2]) || !x.is_cuda()) DECLINE;
  const int dev = x.get_device();
  const ScalarType dt = x.scalar_type();
  if (!plain(x, dev) || !plain(s, dev) || x.dim() != 3 || x.stride(2) != 1 || x.numel() == 0) DECLINE;
  if (!(is_half(dt) || dt == ScalarType::Float) || s.scalar_type() != ScalarType::Float || s.dim() != 1 || s.size(0) != 1) DECLINE;
  const float eps = (float)PyFloat_AS_DOUBLE(a[2]);
  Tensor q;
  {
    Call c(x);
    OBSERVED("mla_quant", x, s);
    q = empty(x.sizes(), ScalarType::Float8_e4m3fn, x.device());
    int32_t* const sync = fp8k_tensor_quant_mla_takes_sync(x.numel()) ? stream_sync(x, c10::hip::getCurrentHIPStream(dev)) : nullptr;
    check(fp8k_tensor_quant_mla_sync(x.data_ptr(), q.data_ptr(), s.data_ptr<float>(), x.size(0), x.size(1), x.size(2), x.stride(0),
                                     x.stride(1), eps, code(dt), sync, c.stream));
  }
  return THPVariable_Wrap(std::move(q));
  END_HANDLE_TH_ERRORS
}

// bmm(A, B, A_scale, B_scale, dtype) -> [b, m, n] or None
PyObject* bmm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor A, B, as, bs;
  if (n != 5 || modes_active() || !tensor_arg(a[0], A) || !tensor_arg(a[1], B) || !tensor_arg(a[2], as) || !tensor_arg(a[3], bs))
    DECLINE;
  if (!THPDtype_Check(a[4]) || !A.is_cuda()) DECLINE;
  const int dev = A.get_device();
  const ScalarType dt = reinterpret_cast<THPDtype*>(a[4])->scalar_type;
  if (!plain(A, dev) || !plain(B, dev) || !plain(as, dev) || !plain(bs, dev) || !is_half(dt) || !is_fp8(A) || !is_fp8(B)) DECLINE;
  if (A.dim() != 3 || B.dim() != 3 || A.size(0) != B.size(0) || A.size(2) != B.size(1) || A.numel() == 0 || B.numel() == 0) DECLINE;
  const int64_t b = A.size(0), m = A.size(1), k = A.size(2), nn = B.size(2);
  if (A.stride(2) != 1 || B.stride(1) != 1 || k % 128 != 0 || nn % 8 != 0) DECLINE;
  if (as.numel() != 1 || bs.numel() != 1 || as.scalar_type() != ScalarType::Float || bs.scalar_type() != ScalarType::Float) DECLINE;
  Tensor out;
  {
    Call c(A);
    OBSERVED("bmm", A, B, as, bs);
    out = empty({b, m, nn}, dt, A.device());
    check(fp8k_bmm_fp8_tensor_scales(A.data_ptr(), B.data_ptr(), as.data_ptr<float>(), bs.data_ptr<float>(), out.data_ptr(), b, m, nn, k,
                       b > 1 ? A.stride(0) : m * k, m > 1 ? A.stride(1) : k, b > 1 ? B.stride(0) : nn * k, nn > 1 ? B.stride(2) : k,
                       m * nn, nn, code(dt), c.stream));
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// ---------------------------------------------------------------------------------------------- experts
// fused_gate(logits, bias, groups, topk_group, topk, shared_experts, scaling, scale_output) -> (weights, ids) or None
PyObject* fused_gate(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor x, bias;
  if (n != 8 || modes_active() || !tensor_arg(a[0], x) || !tensor_arg(a[1], bias) || !x.is_cuda()) DECLINE;
  for (int i = 2; i < 6; ++i)
    if (!PyLong_Check(a[i])) DECLINE;
  if (!PyFloat_Check(a[6])) DECLINE;
  const int dev = x.get_device();
  const ScalarType dt = x.scalar_type();
  if (!plain(x, dev) || !plain(bias, dev) || x.dim() != 2 || bias.dim() != 1 || bias.size(0) != x.size(1) || x.size(0) == 0) DECLINE;
  if (bias.scalar_type() != dt || !(is_half(dt) || dt == ScalarType::Float) || !x.is_contiguous() || !bias.is_contiguous()) DECLINE;
  const int64_t rows = x.size(0), groups = PyLong_AsLongLong(a[2]), topk_group = PyLong_AsLongLong(a[3]);
  const int64_t topk = PyLong_AsLongLong(a[4]), shared = PyLong_AsLongLong(a[5]);
  const double scaling = PyFloat_AS_DOUBLE(a[6]);
  const bool scale_output = truth(a[7]);
  if (topk <= 0 || PyErr_Occurred()) DECLINE;
  Tensor w, ids;
  {
    Call c(x);
    OBSERVED("fused_gate", x, bias);
    w = empty({rows, topk}, ScalarType::Float, x.device());
    ids = empty({rows, topk}, ScalarType::Int, x.device());
    check(fp8k_moe_fused_gate(x.data_ptr(), bias.data_ptr(), w.data_ptr<float>(), ids.data_ptr<int32_t>(), rows, x.size(1), groups,
                              topk_group, topk, shared, scaling, scale_output ? 1 : 0, code(dt), c.stream));
  }
  PyObject* out = PyTuple_New(2);
  if (!out) return nullptr;
  PyTuple_SET_ITEM(out, 0, THPVariable_Wrap(std::move(w)));
  PyTuple_SET_ITEM(out, 1, THPVariable_Wrap(std::move(ids)));
  return out;
  END_HANDLE_TH_ERRORS
}

// expert weights: w e4m3fn [E, rows, K] contiguous, scale float32 [E, ceil(rows/128), K/128]
bool expert_weight(const Tensor& w, const Tensor& s, int dev) {
  if (!plain(w, dev) || !plain(s, dev) || !is_fp8(w) || w.dim() != 3 || !w.is_contiguous() || w.numel() == 0) return false;
  return s.scalar_type() == ScalarType::Float && s.dim() == 3 && non_negative_strides(s) && s.size(0) == w.size(0) &&
         s.size(1) == ceil_div(w.size(1), 128) && s.size(2) == ceil_div(w.size(2), 128) && w.size(2) % 128 == 0;
}

// fused_experts(x, w13, w2, w13_scale, w2_scale, topk_weights, topk_ids, block_m, balanced, fuse_gemm1, weight_on_input,
//               scaling, inplace) -> output or None: the gated silu experts of fused_moe.fused_experts_impl in one call.  The
// decisions (block_m, balanced, fuse_gemm1) are the Python side's.
PyObject* fused_experts(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor x, w13, w2, s13, s2, tw, ids;
  if (n != 13 || modes_active() || !tensor_arg(a[0], x) || !tensor_arg(a[1], w13) || !tensor_arg(a[2], w2) || !tensor_arg(a[3], s13) ||
      !tensor_arg(a[4], s2) || !tensor_arg(a[5], tw) || !tensor_arg(a[6], ids) || !x.is_cuda())
    DECLINE;
  if (!PyLong_Check(a[7]) || !PyFloat_Check(a[11])) DECLINE;
  const int64_t bm = PyLong_AsLongLong(a[7]);
  const bool balanced = truth(a[8]), fuse = truth(a[9]), on_input = truth(a[10]), inplace = truth(a[12]);
  const int dev = x.get_device();
  const ScalarType dt = x.scalar_type();
  if (!plain(x, dev) || !is_half(dt) || x.dim() != 2 || x.numel() == 0 || !x.is_contiguous()) DECLINE;
  if (!expert_weight(w13, s13, dev) || !expert_weight(w2, s2, dev)) DECLINE;
  const int64_t T = x.size(0), H = x.size(1), E = w13.size(0), N = w13.size(1), I = N / 2;
  if (w13.size(2) != H || w2.size(0) != E || w2.size(1) != H || w2.size(2) != I || N % 256 != 0 || H % 128 != 0) DECLINE;
  if (!plain(tw, dev) || !plain(ids, dev) || tw.dim() != 2 || ids.dim() != 2 || tw.sizes() != ids.sizes() || ids.size(0) != T) DECLINE;
  if (tw.scalar_type() != ScalarType::Float || !tw.is_contiguous() || !ids.is_contiguous()) DECLINE;
  const bool ids64 = ids.scalar_type() == ScalarType::Long;
  if (!ids64 && ids.scalar_type() != ScalarType::Int) DECLINE;
  const int64_t topk = ids.size(1), slots = T * topk;
  if (topk <= 0 || bm <= 0 || (fuse && (bm != 256 || on_input)) || (balanced && bm != 256)) DECLINE;

  const int64_t cap = slots + (E + 1) * (bm - 1), blocks = ceil_div(cap, bm);
  // what of the table can be in use (a block holds at least one slot, and only an expert's last is not full): the launches
  // are sized by it, 7168 workgroups less for 2 tokens of 128 experts
  const int64_t cap_used = std::min(cap, bm * std::min(slots, E + 1 + slots / bm));
  const int64_t kb1 = H / 128, kb2 = I / 128;
  const bool act_gemm2 = !fuse && fp8k_moe_act_block_gemm_takes(bm, H, I, I);  // silu_and_mul and requantisation inside GEMM 2
  const bool sorted = bm >= 64;  // blocks of 64 slots and more read their activation scales in slot order
  const float scaling = (float)PyFloat_AS_DOUBLE(a[11]);
  Tensor out;
  {
    Call c(x);
    OBSERVED("fused_experts", x, w13, w2, s13, s2, tw, ids);
    out = inplace ? x : empty(x.sizes(), dt, x.device());
    const int64_t b_ids = cap * 4, b_q1 = T * H, b_s1 = T * kb1 * 4, b_ss1 = cap * kb1 * 4, b_mid = slots * N * 2, b_q2 = slots * I,
                  b_s2 = slots * kb2 * 4, b_ss2 = cap * kb2 * 4, b_out = slots * H * 2;
    using S = Scratch;
    Scratch mem(2 * S::room(b_ids) + S::room(blocks * 4) + S::room(4) + S::room((E + 2) * 4) + S::room(b_q1) + S::room(b_s1) +
                    (sorted ? S::room(b_ss1) + S::room(b_ss2) : 0) + (fuse ? 0 : S::room(b_mid) + S::room(b_s2)) + S::room(b_q2) +
                    S::room(b_out),
                c.stream);
    int32_t* sorted_ids = mem.take<int32_t>(b_ids);
    int32_t* even_ids = mem.take<int32_t>(b_ids);
    int32_t* block_expert = mem.take<int32_t>(blocks * 4);
    int32_t* padded = mem.take<int32_t>(4);
    int32_t* cumsum = mem.take<int32_t>((E + 2) * 4);
    void* q1 = mem.take(b_q1);
    float* s1 = mem.take<float>(b_s1);
    void* q2 = mem.take(b_q2);
    void* down = mem.take(b_out);
    float* ss1 = sorted ? mem.take<float>(b_ss1) : nullptr;
    float* ss2 = sorted ? mem.take<float>(b_ss2) : nullptr;
    void* mid = fuse ? nullptr : mem.take(b_mid);
    float* sm2 = fuse ? nullptr : mem.take<float>(b_s2);
    const int dc = code(dt);
    const float* twp = tw.data_ptr<float>();
    void* st = c.stream;

    // small blocks read their scales column-major per token, large ones get them gathered into slot order
    check(fp8k_moe_align_quant(ids.data_ptr(), ids64, slots, E + 1, bm, sorted_ids, cap, block_expert, blocks, padded, cumsum, x.data_ptr(), q1,
                               s1, T, H, kEps, dc, sorted ? kb1 : 1, sorted ? 1 : T, st));
    if (balanced) {
      check(fp8k_moe_balance_blocks(sorted_ids, block_expert, padded, cap, bm, slots, E, even_ids, st));
      sorted_ids = even_ids;
    }
    if (sorted) check(fp8k_moe_sort_scales(s1, ss1, sorted_ids, padded, cap, kb1, topk, slots, kb1, 1, st));
    auto gemm = [&](const void* A, const Tensor& W, const Tensor& Ws, const float* As, int64_t as_m, int64_t as_k, void* C, bool weigh,
                    int64_t per_row) {
      check(fp8k_moe_block_gemm(A, W.data_ptr(), As, Ws.data_ptr<float>(), C, sorted_ids, block_expert, padded, weigh ? twp : nullptr, cap_used,
                                bm, slots, per_row, E, W.size(1), W.size(2), W.size(2), as_m, as_k, W.stride(0), W.stride(1), Ws.stride(0),
                                Ws.stride(1), Ws.stride(2), W.size(1), dc, (sorted ? 1 : 0) | (balanced ? 2 : 0), st));
    };
    if (fuse) {
      check(fp8k_moe_block_gemm_silu_quant(q1, w13.data_ptr(), ss1, s13.data_ptr<float>(), q2, ss2, sorted_ids, block_expert, padded, cap,
                                           slots, topk, E, N, H, H, cap, w13.stride(0), w13.stride(1), s13.stride(0), s13.stride(1),
                                           s13.stride(2), I, cap, kEps, dc, balanced ? 1 : 0, st));
    } else {
      gemm(q1, w13, s13, sorted ? ss1 : s1, 1, sorted ? cap : T, mid, on_input, topk);
    }
    if (act_gemm2) {
      check(fp8k_moe_act_block_gemm(mid, w2.data_ptr(), s2.data_ptr<float>(), down, sorted_ids, block_expert, padded, on_input ? nullptr : twp,
                                    cap_used, bm, slots, E, H, I, N, w2.stride(0), I, s2.stride(0), s2.stride(1), s2.stride(2), H, kEps, dc, st));
    } else if (!fuse) {
      check(fp8k_silu_mul_group_quant(mid, q2, sm2, slots, I, 128, kEps, -448.f, 448.f, dc, sorted ? kb2 : 1, sorted ? 1 : slots,
                                      FP8K_SCALE_F32, st));
      if (sorted) check(fp8k_moe_sort_scales(sm2, ss2, sorted_ids, padded, cap, kb2, 1, slots, kb2, 1, st));
    }
    if (!act_gemm2) gemm(q2, w2, s2, sorted ? ss2 : sm2, 1, sorted ? cap : slots, down, !on_input, 1);
    check(fp8k_moe_sum_reduce(down, out.data_ptr(), T, topk, H, topk * H, H, H, scaling, dc, st));
  }
  if (inplace) {
    Py_INCREF(a[0]);
    return a[0];
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// set_workspace(registry, grow): the per-stream GEMM workspaces of sgl_kernel
PyObject* set_workspace(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 2 || !PyDict_Check(a[0]) || !PyCallable_Check(a[1])) {
    PyErr_SetString(PyExc_TypeError, "set_workspace(dict, callable)");
    return nullptr;
  }
  Py_INCREF(a[0]);
  Py_INCREF(a[1]);
  g_workspaces = a[0];
  g_grow_workspace = a[1];
  Py_RETURN_NONE;
}

#define FN(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {FN(group_quant), FN(block_linear), FN(block_matmul), FN(token_linear), FN(mla_quant),     FN(bmm),
                         FN(fused_gate),  FN(fused_experts), FN(set_workspace), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", "native calls of the layer-level entry points", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) {
  PyObject* const overrides = PyImport_ImportModule("torch.overrides");
  if (!overrides) return nullptr;
  g_has_torch_function = PyObject_GetAttrString(overrides, "has_torch_function_unary");
  Py_DECREF(overrides);
  if (!g_has_torch_function) return nullptr;
  PyObject* const m = PyModule_Create(&module);
  if (m && PyModule_AddStringConstant(m, "torch", FP8K_TORCH_MARK) < 0) return nullptr;
  return m;
}
