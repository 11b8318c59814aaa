// The host path of the operators that a model calls once per layer and step: argument checks,
// outputs, scratch, stream, and the calls into libsglq, in one C++ call per operator.
//
// What bounds a decode-sized call is this path, not the GPU: through ctypes a linear of one to a few
// hundred rows took 17-37 us of Python (two launches of together 5-25 us on the GPU), most of it tensor
// properties read one attribute at a time, views (`.T`, `.view`), three `torch.empty`, two trips through
// the dispatcher and the conversion of 18 arguments per ctypes call.  From here: 1 x 2112 x 7168 block-FP8
// linear 17.4 -> 8.0 us a pass (GPU-bound now), 16 x 14336 x 4096 INT8 with bias 26.2 -> 16.0, the two
// operators on 333 x 4096 x 7168 35.5 -> 28.7, small shapes 25-36 -> 7-13.
//
// Every function here takes exactly the calls that need no conversion and no error message: tensors on
// the GPU in the layouts the kernels read.  For anything else (another layout, a shape or dtype that the
// operator refuses, a call that autograd, a transform, a mode or a profiler has to see) it returns None, and
// the Python function it was called from composes the same operators with torch or raises: argument rules are
// therefore here and there, and only Python's carry messages.
//
// The library's entry points arrive as addresses (`bind`), so that the shared object that `_lib.load()`
// opened is the one that runs.
#include <Python.h>

#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/grad_mode.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/ops/add.h>
#include <ATen/ops/fill.h>
#include <ATen/record_function.h>
#include <c10/core/DispatchKeySet.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <iterator>
#include <memory>
#include <mutex>
#include <unordered_map>
#include <vector>

#include "../../include/sglq.h"

namespace {

// ---------------------------------------------------------------------------
// the library's entry points
// ---------------------------------------------------------------------------
#define SGLQ_HOST_ENTRY_POINTS(X)                                                                                   \
  X(sglq_per_token_group_quant_fp8)                                                                                 \
  X(sglq_per_token_group_quant_int8)                                                                                \
  X(sglq_per_token_group_quant_fp8_pow2)                                                                            \
  X(sglq_per_token_quant_fp8)                                                                                       \
  X(sglq_per_token_quant_int8)                                                                                      \
  X(sglq_fp8_blockwise_scaled_mm)                                                                                   \
  X(sglq_fp8_blockwise_scaled_mm_bias)                                                                              \
  X(sglq_fp8_blockwise_scaled_mm_ue8m0)                                                                             \
  X(sglq_int8_blockwise_scaled_mm)                                                                                  \
  X(sglq_int8_blockwise_scaled_mm_bias)                                                                             \
  X(sglq_int8_scaled_mm)                                                                                            \
  X(sglq_fp8_scaled_mm)                                                                                             \
  X(sglq_prepare_moe_input)                                                                                         \
  X(sglq_prepare_moe_layer)                                                                                         \
  X(sglq_prepare_moe_layer_rows)                                                                                    \
  X(sglq_prepare_moe_layer_walks)                                                                                   \
  X(sglq_prepare_moe_layer_quant)                                                                                   \
  X(sglq_fp8_blockwise_scaled_grouped_mm_silu_few_rows)                                                                   \
  X(sglq_grouped_few_rows_activates)                                                                                \
  X(sglq_grouped_gathers)                                                                                           \
  X(sglq_grouped_walk_bytes)                                                                                        \
  X(sglq_grouped_layer_rows)                                                                                        \
  X(sglq_fp8_blockwise_scaled_grouped_mm_tiled)                                                                     \
  X(sglq_fp8_blockwise_scaled_grouped_mm_walked)                                                                    \
  X(sglq_fp8_blockwise_scaled_grouped_mm_silu)                                                                      \
  X(sglq_fp8_blockwise_scaled_grouped_mm_gathered)                                                                  \
  X(sglq_grouped_plan_rows)                                                                                         \
  X(sglq_fp8_blockwise_scaled_grouped_mm)                                                                           \
  X(sglq_fp8_blockwise_scaled_grouped_mm_planned)                                                                   \
  X(sglq_per_token_group_quant_fp8_scatter_cm)                                                                      \
  X(sglq_per_token_group_quant_fp8_scatter_scales_cm)                                                               \
  X(sglq_silu_and_mul_group_quant_fp8_cm)                                                                           \
  X(sglq_apply_shuffle_mul_sum)                                                                                     \
  X(sglq_apply_shuffle_mul_sum_f32)                                                                                 \
  X(sglq_w8a8_block_fp8_linear)                                                                                     \
  X(sglq_w8a8_int8_linear)                                                                                          \
  X(sglq_w8a8_fp8_linear)

struct EntryPoints {
#define X(name) decltype(&::name) name = nullptr;
  SGLQ_HOST_ENTRY_POINTS(X)
#undef X
};
EntryPoints lib;
bool bound = false;

// ---------------------------------------------------------------------------
// scratch: kept per device and stream, so that two streams never share it; a mutex per buffer keeps the
// launches of one operator together when two threads use one stream
// ---------------------------------------------------------------------------
constexpr int64_t SPLITK_BYTES = 64 << 20;  // what the GEMMs' selection rules were measured with
// Quantized activations in front of it: kept for the sizes where an allocation would be felt (16 MiB is
// 4096 rows of 4096, or 512 rows of 28672), allocated per call above.
constexpr int64_t CODES_BYTES = (16 << 20) + (1 << 20);
constexpr size_t MAX_WORKSPACES = 64;  // beyond as many (device, stream) pairs scratch is allocated per call

struct Workspace {
  at::Tensor buffer;
  char* base = nullptr;
  std::mutex lock;
};

struct StreamKey {
  int device;
  void* stream;
  bool operator==(const StreamKey& o) const { return device == o.device && stream == o.stream; }
};
struct StreamKeyHash {
  size_t operator()(const StreamKey& k) const { return std::hash<void*>()(k.stream) * 31 + (size_t)k.device; }
};
using Workspaces = std::unordered_map<StreamKey, std::shared_ptr<Workspace>, StreamKeyHash>;
std::mutex workspaces_lock;
Workspaces& workspaces = *new Workspaces;  // (never destroyed: at process exit torch's allocator may be gone first)

at::Tensor empty(at::IntArrayRef sizes, at::ScalarType dtype, c10::Device device) {
  return at::detail::empty_cuda(sizes, dtype, device, std::nullopt);
}

std::shared_ptr<Workspace> workspace_of(c10::Device device, void* stream) {
  std::lock_guard<std::mutex> guard(workspaces_lock);
  auto it = workspaces.find(StreamKey{device.index(), stream});
  if (it != workspaces.end()) return it->second;
  auto w = std::make_shared<Workspace>();
  w->buffer = empty({CODES_BYTES + SPLITK_BYTES}, at::kByte, device);
  w->base = static_cast<char*>(w->buffer.data_ptr());
  if (workspaces.size() < MAX_WORKSPACES) workspaces.emplace(StreamKey{device.index(), stream}, w);
  return w;
}

bool capturing(void* stream) {
  if (stream == nullptr) return false;  // (the default stream cannot be captured)
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(static_cast<hipStream_t>(stream), &status) != hipSuccess) {
    (void)hipGetLastError();  // (the launches that follow report what is wrong with the stream)
    return false;
  }
  return status != hipStreamCaptureStatusNone;
}

// What one operator call writes its codes and scales to (`codes`, `codes_bytes` of them) and, behind them or
// apart, its split-K partial sums.  Under capture all of it is allocated by the call, from the graph's own pool:
// a graph keeps the addresses for its replays, and two graphs that were captured on one stream (torch captures
// all of them on one unless told otherwise) may be replayed at the same time on two.
struct Scratch {
  at::Tensor own;  // freed when the call returns; what reuses the memory is ordered behind it on the stream
  std::shared_ptr<Workspace> kept;
  std::unique_lock<std::mutex> one_operator;
  char* codes = nullptr;
  char* partial = nullptr;
  int64_t partial_bytes = SPLITK_BYTES;

  // m, n, k: the GEMM's.  Its K is split in at most as many parts as it has blocks of 128, so that a capture's
  // smaller piece leads to the same choice of kernel and split as the kept one.
  Scratch(c10::Device device, void* stream, int64_t codes_bytes, int64_t m, int64_t n, int64_t k) {
    if (capturing(stream)) {
      const int64_t sums = (4 * m * n * ((k + 127) / 128) + 255) & ~int64_t(255);
      if (sums < partial_bytes) partial_bytes = sums;
      own = empty({codes_bytes + partial_bytes}, at::kByte, device);
      codes = static_cast<char*>(own.data_ptr());
      partial = codes + codes_bytes;
      return;
    }
    kept = workspace_of(device, stream);
    if (codes_bytes > CODES_BYTES) {
      own = empty({codes_bytes}, at::kByte, device);
      codes = static_cast<char*>(own.data_ptr());
      partial = kept->base;
    } else {
      codes = kept->base;
      partial = codes + codes_bytes;
    }
    one_operator = std::unique_lock<std::mutex>(kept->lock);
  }
  bool in_one_piece(int64_t codes_bytes) const { return partial == codes + codes_bytes; }
};

// ---------------------------------------------------------------------------
// arguments
// ---------------------------------------------------------------------------
using at::Tensor;

constexpr auto FP8 = at::kFloat8_e4m3fn;

inline int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kBFloat16: return SGLQ_BF16;
    case at::kHalf: return SGLQ_FP16;
    case at::kFloat: return SGLQ_FP32;
    default: return -1;
  }
}
inline bool is_16bit(at::ScalarType t) { return t == at::kBFloat16 || t == at::kHalf; }

// A plain tensor (or Parameter) on the GPU; subclasses with behaviour of their own stay with Python.
inline const Tensor* gpu_tensor(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const Tensor& t = THPVariable_Unpack(o);
  return t.is_cuda() && t.layout() == at::kStrided ? &t : nullptr;
}
inline bool optional_tensor(PyObject* o, const Tensor*& t) {
  t = nullptr;
  if (o == Py_None) return true;
  t = gpu_tensor(o);
  return t != nullptr;
}

// Whether a call may go past torch's dispatcher: the tensors are what they seem (no functorch level, no lazy negation or
// conjugation, nothing but a strided GPU tensor with or without autograd), no one is watching (torch.jit.trace, vmap and
// the other transforms, dispatch and function modes, a profiler's callbacks), nothing needs a gradient.
constexpr c10::DispatchKeySet PLAIN_KEYS = c10::DispatchKeySet(c10::BackendComponent::CUDABit) |
                                           c10::DispatchKeySet({c10::DispatchKey::Dense, c10::DispatchKey::ADInplaceOrView}) |
                                           c10::autograd_dispatch_keyset | c10::autocast_dispatch_keyset;
inline bool plain(const Tensor& t) {
  return (t.key_set().raw_repr() & ~PLAIN_KEYS.raw_repr()) == 0 && !(at::GradMode::is_enabled() && t.requires_grad());
}
inline bool watched() {
  return !(c10::impl::tls_local_dispatch_key_set().included_ - c10::default_included_set).empty() ||
         c10::impl::dispatch_mode_enabled() || at::impl::torch_function_mode_enabled() || at::hasCallbacks();
}
template <typename... T>
inline bool direct(const T&... tensors) {
  return bound && !watched() && (... && plain(tensors));
}
inline bool plain(const Tensor* t) { return t == nullptr || plain(*t); }

// Current stream and, where the tensors live on another GPU than the current one, that GPU made current.
struct Launch {
  c10::Device device;
  c10::DeviceIndex previous = -1;
  void* stream;
  explicit Launch(c10::Device d) : device(d) {
    const c10::DeviceIndex current = c10::hip::current_device();
    if (current != d.index()) {
      previous = current;
      c10::hip::set_device(d.index());
    }
    stream = static_cast<void*>(c10::hip::getCurrentHIPStream(d.index()).stream());
  }
  ~Launch() {
    if (previous >= 0) c10::hip::set_device(previous);
  }
};

struct ReleaseGil {
  PyThreadState* state;
  ReleaseGil() : state(PyEval_SaveThread()) {}
  ~ReleaseGil() { PyEval_RestoreThread(state); }
};

inline int64_t round256(int64_t v) { return (v + 255) & ~int64_t(255); }

inline PyObject* none() { Py_RETURN_NONE; }

// [..., K] -> [..., n]
inline std::vector<int64_t> output_shape(const Tensor& x, int64_t n) {
  std::vector<int64_t> s(x.sizes().begin(), x.sizes().end());
  s.back() = n;
  return s;
}

// C++ exceptions (the allocator's out-of-memory among them) become torch's Python errors.
template <typename F>
PyObject* guarded(F&& body) {
  HANDLE_TH_ERRORS
  return body();
  END_HANDLE_TH_ERRORS
}

inline bool aligned(const Tensor& t, uintptr_t bytes) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & (bytes - 1)) == 0; }

// Activations [..., K] as the quantization kernels read them.
inline bool activations(const Tensor& x) {
  return is_16bit(x.scalar_type()) && x.dim() >= 1 && x.is_contiguous() && x.numel() > 0 && aligned(x, 16);
}
inline bool bias_fits(const Tensor* bias, int64_t n, at::ScalarType dtype, const Tensor& like) {
  return bias == nullptr || (bias->scalar_type() == dtype && bias->is_contiguous() && bias->numel() == n && bias->device() == like.device());
}

// ---------------------------------------------------------------------------
// block-scaled linears: x [..., K], weight [N, K] as stored, weight_scale [ceil(N/128), K/128]
// ---------------------------------------------------------------------------
enum BlockMode { BLOCK_FP8 = 0, BLOCK_FP8_POW2 = 1, BLOCK_INT8 = 2 };

// Weight scales that have been checked to be powers of two (check_pow2_scales in quantization/fp8_kernel.py): storage,
// place in it, shape, strides and version counter.  The weak reference keeps the storage's own address from being used
// again, so that what a new tensor at an old address holds is not taken for checked.
struct ScalesKey {
  const c10::StorageImpl* storage;
  const void* ptr;
  int64_t rows, cols, stride_r, stride_c;
  uint32_t version;
  bool operator==(const ScalesKey& o) const {
    return storage == o.storage && ptr == o.ptr && rows == o.rows && cols == o.cols && stride_r == o.stride_r && stride_c == o.stride_c &&
           version == o.version;
  }
};
struct ScalesKeyHash {
  size_t operator()(const ScalesKey& k) const { return std::hash<const void*>()(k.ptr) * 31 + k.version; }
};
constexpr size_t MAX_CHECKED_SCALES = 4096;
std::mutex checked_lock;
auto& checked_scales = *new std::unordered_map<ScalesKey, c10::weak_intrusive_ptr<c10::StorageImpl>, ScalesKeyHash>;

inline ScalesKey scales_key(const Tensor& t) {
  return {t.storage().unsafeGetStorageImpl(), t.const_data_ptr(), t.size(0), t.size(1), t.stride(0), t.stride(1), (uint32_t)t._version()};
}
inline bool pow2_checked(const Tensor& t) {
  std::lock_guard<std::mutex> guard(checked_lock);
  return checked_scales.find(scales_key(t)) != checked_scales.end();
}
// (an inference tensor has no version counter: in-place changes would go unseen)
inline const Tensor* versioned_matrix(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const Tensor& t = THPVariable_Unpack(o);
  return t.layout() == at::kStrided && t.dim() == 2 && t.has_storage() && !t.is_inference() ? &t : nullptr;
}

PyObject* pow2_scales_known(PyObject*, PyObject* arg) {
  return guarded([&]() -> PyObject* {
    const Tensor* t = versioned_matrix(arg);
    return PyBool_FromLong(t && pow2_checked(*t));
  });
}
PyObject* note_pow2_scales(PyObject*, PyObject* arg) {
  return guarded([&]() -> PyObject* {
    if (const Tensor* t = versioned_matrix(arg)) {
      std::lock_guard<std::mutex> guard(checked_lock);
      if (checked_scales.size() >= MAX_CHECKED_SCALES) {
        for (auto it = checked_scales.begin(); it != checked_scales.end();) it = it->second.expired() ? checked_scales.erase(it) : std::next(it);
        if (checked_scales.size() >= MAX_CHECKED_SCALES) checked_scales.clear();
      }
      checked_scales.insert_or_assign(scales_key(*t), t->storage().getWeakStorageImpl());
    }
    return none();
  });
}

// block_linear(x, weight, weight_scale, bias | None, mode, eps) -> [..., N]
PyObject* block_linear(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 6) return PyErr_Format(PyExc_TypeError, "block_linear takes 6 arguments");
  return guarded([&]() -> PyObject* {
    const Tensor *xp = gpu_tensor(args[0]), *wp = gpu_tensor(args[1]), *sp = gpu_tensor(args[2]), *bias;
    if (!xp || !wp || !sp || !optional_tensor(args[3], bias)) return none();
    const long mode = PyLong_AsLong(args[4]);
    const float eps = (float)PyFloat_AsDouble(args[5]);
    const Tensor &x = *xp, &w = *wp, &s = *sp;
    if (!direct(x, w, s) || !plain(bias)) return none();
    if (!activations(x) || w.dim() != 2 || s.dim() != 2 || !w.is_contiguous() || s.scalar_type() != at::kFloat) return none();
    if (w.scalar_type() != (mode == BLOCK_INT8 ? at::kChar : FP8)) return none();
    const int64_t k = x.size(-1), m = x.numel() / k, n = w.size(0), kb = k / 128;
    if (w.size(1) != k || k % 128 != 0 || n % 8 != 0 || n == 0 || s.size(0) != (n + 127) / 128 || s.size(1) != kb) return none();
    if (s.stride(1) != 1 && kb > 1) return none();
    if (w.device() != x.device() || s.device() != x.device() || !aligned(w, 16)) return none();
    const at::ScalarType dtype = x.scalar_type();
    if (!bias_fits(bias, n, dtype, x)) return none();
    if (mode == BLOCK_FP8_POW2) {
      if (dtype != at::kBFloat16 || n % 64 != 0 || s.is_inference() || !pow2_checked(s)) return none();
    }
    const int64_t need = round256(m * k) + round256(m * kb * 4);
    Tensor out;
    int rc;
    {
      ReleaseGil unlocked;
      Launch here(x.device());
      out = empty(output_shape(x, n), dtype, here.device);
      Scratch scratch(here.device, here.stream, need, m, n, k);
      void* const partial = scratch.partial;
      const int64_t partial_bytes = scratch.partial_bytes;
      const int code = dtype_code(dtype);
      void* out_p = out.data_ptr();
      const void *x_p = x.data_ptr(), *w_p = w.data_ptr(), *bias_p = bias ? bias->data_ptr() : nullptr;
      const float* s_p = static_cast<const float*>(s.data_ptr());
      const int64_t sn = s.stride(0);
      if (mode == BLOCK_FP8 && scratch.in_one_piece(need)) {
        rc = lib.sglq_w8a8_block_fp8_linear(x_p, code, w_p, k, s_p, 1, sn, bias_p, out_p, n, code, m, n, k, eps, scratch.codes,
                                            need + partial_bytes, here.stream);
      } else {
        char* codes = scratch.codes;
        float* scales = reinterpret_cast<float*>(codes + round256(m * k));
        if (mode == BLOCK_INT8) {
          // (column-major scales: the GEMM fetches a K block's scales of 64 rows with one instruction, from two cache
          // lines instead of up to 64; 1000 x 5120 x 5120 with bias 49.8 -> 42 us together with gemm_ring_kernel)
          rc = lib.sglq_per_token_group_quant_int8(x_p, code, codes, scales, m, k, 128, 1, m, eps, -128.0f, 127.0f, here.stream);
          if (rc == 0 && bias_p)
            rc = lib.sglq_int8_blockwise_scaled_mm_bias(codes, k, w_p, k, scales, 1, m, s_p, 1, sn, bias_p, out_p, n, code, m, n, k, partial,
                                                        partial_bytes, here.stream);
          else if (rc == 0)
            rc = lib.sglq_int8_blockwise_scaled_mm(codes, k, w_p, k, scales, 1, m, s_p, 1, sn, out_p, n, code, m, n, k, partial, partial_bytes,
                                                   here.stream);
        } else if (mode == BLOCK_FP8_POW2) {
          rc = lib.sglq_per_token_group_quant_fp8_pow2(x_p, code, codes, scales, m, k, 1, m, eps, -448.0f, 448.0f, here.stream);
          if (rc == 0)
            rc = lib.sglq_fp8_blockwise_scaled_mm_ue8m0(codes, k, w_p, k, scales, 1, m, s_p, 1, sn, out_p, n, code, m, n, k, partial,
                                                        partial_bytes, here.stream);
        } else {
          rc = lib.sglq_per_token_group_quant_fp8(x_p, code, codes, scales, m, k, 128, 1, m, eps, -448.0f, 448.0f, here.stream);
          if (rc == 0 && bias_p)
            rc = lib.sglq_fp8_blockwise_scaled_mm_bias(codes, k, w_p, k, scales, 1, m, s_p, 1, sn, bias_p, out_p, n, code, m, n, k, partial,
                                                       partial_bytes, here.stream);
          else if (rc == 0)
            rc = lib.sglq_fp8_blockwise_scaled_mm(codes, k, w_p, k, scales, 1, m, s_p, 1, sn, out_p, n, code, m, n, k, partial, partial_bytes,
                                                  here.stream);
        }
      }
      if (rc == 0 && bias && mode == BLOCK_FP8_POW2) {
        at::NoGradGuard no_grad;
        out.add_(*bias);
      }
    }
    return rc == 0 ? THPVariable_Wrap(std::move(out)) : none();
  });
}

// token_linear(x, weight_kn, weight_scale, bias | None, is_int8) -> [..., N]: per-token activation scales,
// per-channel weight scales; weight_kn [K, N] column-major
PyObject* token_linear(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 5) return PyErr_Format(PyExc_TypeError, "token_linear takes 5 arguments");
  return guarded([&]() -> PyObject* {
    const Tensor *xp = gpu_tensor(args[0]), *wp = gpu_tensor(args[1]), *sp = gpu_tensor(args[2]), *bias;
    if (!xp || !wp || !sp || !optional_tensor(args[3], bias)) return none();
    const bool int8 = args[4] == Py_True;
    const Tensor &x = *xp, &w = *wp, &s = *sp;
    if (!direct(x, w, s) || !plain(bias)) return none();
    if (!activations(x) || w.dim() != 2 || w.stride(0) != 1 || w.scalar_type() != (int8 ? at::kChar : FP8)) return none();
    const int64_t k = x.size(-1), m = x.numel() / k, n = w.size(1);
    if (w.size(0) != k || k % 16 != 0 || n % 8 != 0 || n <= 1) return none();
    const int64_t ldb = w.stride(1);
    if (ldb % 16 != 0 || ldb < k || !aligned(w, 16)) return none();
    if (s.scalar_type() != at::kFloat || !s.is_contiguous() || s.numel() != n || !aligned(s, 16)) return none();
    if (w.device() != x.device() || s.device() != x.device()) return none();
    const at::ScalarType dtype = x.scalar_type();
    if (!bias_fits(bias, n, dtype, x)) return none();
    const int64_t need = round256(m * k) + round256(m * 4);
    Tensor out;
    int rc;
    {
      ReleaseGil unlocked;
      Launch here(x.device());
      out = empty(output_shape(x, n), dtype, here.device);
      Scratch scratch(here.device, here.stream, need, m, n, k);
      const int code = dtype_code(dtype);
      const void *x_p = x.data_ptr(), *w_p = w.data_ptr(), *bias_p = bias ? bias->data_ptr() : nullptr;
      const float* s_p = static_cast<const float*>(s.data_ptr());
      if (scratch.in_one_piece(need)) {
        rc = (int8 ? lib.sglq_w8a8_int8_linear : lib.sglq_w8a8_fp8_linear)(x_p, code, w_p, ldb, s_p, bias_p, out.data_ptr(), n, code, m, n, k,
                                                                           scratch.codes, need + scratch.partial_bytes, here.stream);
      } else {
        char* codes = scratch.codes;
        float* scales = reinterpret_cast<float*>(codes + round256(m * k));
        rc = int8 ? lib.sglq_per_token_quant_int8(x_p, code, codes, scales, nullptr, m, k, here.stream)
                  : lib.sglq_per_token_quant_fp8(x_p, code, codes, scales, m, k, here.stream);
        if (rc == 0)
          rc = (int8 ? lib.sglq_int8_scaled_mm : lib.sglq_fp8_scaled_mm)(codes, k, w_p, ldb, scales, s_p, bias_p, out.data_ptr(), n, code, m, n, k,
                                                                         scratch.partial, scratch.partial_bytes, here.stream);
      }
    }
    return rc == 0 ? THPVariable_Wrap(std::move(out)) : none();
  });
}

// ---------------------------------------------------------------------------
// the operators one by one
// ---------------------------------------------------------------------------
inline bool out_dtype_of(PyObject* o, at::ScalarType& t) {
  if (!THPDtype_Check(o)) return false;
  t = reinterpret_cast<THPDtype*>(o)->scalar_type;
  return is_16bit(t);
}

// What the three GEMM operators ask of their operands (check_mm_common in sgl_kernel/gemm.py).
inline bool mm_operands(const Tensor& a, const Tensor& b, at::ScalarType elem) {
  if (a.dim() != 2 || b.dim() != 2 || a.scalar_type() != elem || b.scalar_type() != elem) return false;
  const int64_t m = a.size(0), k = a.size(1), n = b.size(1);
  if (m == 0 || n == 0 || k == 0 || b.size(0) != k || k % 16 != 0 || n % 8 != 0) return false;
  if (a.stride(1) != 1 || b.stride(0) != 1 || (m > 1 && a.stride(0) % 16 != 0) || (n > 1 && b.stride(1) % 16 != 0)) return false;
  return a.device() == b.device();
}
inline bool vector_like(const Tensor& t) {
  return t.is_contiguous() && (t.dim() == 1 || (t.dim() == 2 && (t.size(0) == 1 || t.size(1) == 1)));
}

// blockwise_mm(a, b, scales_a, scales_b, out_dtype, bias | None, dispatched) -> [M, N]
// `dispatched`: called from the operator's implementation, behind torch's dispatcher.
PyObject* blockwise_mm(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 7) return PyErr_Format(PyExc_TypeError, "blockwise_mm takes 7 arguments");
  return guarded([&]() -> PyObject* {
    const Tensor *ap = gpu_tensor(args[0]), *bp = gpu_tensor(args[1]), *sap = gpu_tensor(args[2]), *sbp = gpu_tensor(args[3]), *bias;
    at::ScalarType dtype;
    if (!ap || !bp || !sap || !sbp || !optional_tensor(args[5], bias) || !out_dtype_of(args[4], dtype)) return none();
    const Tensor &a = *ap, &b = *bp, &sa = *sap, &sb = *sbp;
    if (!bound || (args[6] != Py_True && (!direct(a, b, sa, sb) || !plain(bias)))) return none();
    if (!mm_operands(a, b, FP8)) return none();
    const int64_t m = a.size(0), k = a.size(1), n = b.size(1), kb = (k + 127) / 128, nb = (n + 127) / 128;
    if (sa.scalar_type() != at::kFloat || sb.scalar_type() != at::kFloat || sa.dim() != 2 || sb.dim() != 2) return none();
    if (sa.size(0) != m || sa.size(1) != kb || sb.size(0) != kb || sb.size(1) != nb) return none();
    if ((sa.stride(0) != 1 && !vector_like(sa)) || (sb.stride(0) != 1 && !vector_like(sb))) return none();
    if (sa.device() != a.device() || sb.device() != a.device() || !bias_fits(bias, n, dtype, a)) return none();
    Tensor out;
    int rc;
    {
      ReleaseGil unlocked;
      Launch here(a.device());
      out = empty({m, n}, dtype, here.device);
      Scratch scratch(here.device, here.stream, 0, m, n, k);
      const int64_t lda = m > 1 ? a.stride(0) : k, ldb = n > 1 ? b.stride(1) : k;
      const float *sa_p = static_cast<const float*>(sa.data_ptr()), *sb_p = static_cast<const float*>(sb.data_ptr());
      if (bias)
        rc = lib.sglq_fp8_blockwise_scaled_mm_bias(a.data_ptr(), lda, b.data_ptr(), ldb, sa_p, sa.stride(0), sa.stride(1), sb_p, sb.stride(0),
                                                   sb.stride(1), bias->data_ptr(), out.data_ptr(), n, dtype_code(dtype), m, n, k,
                                                   scratch.partial, scratch.partial_bytes, here.stream);
      else
        rc = lib.sglq_fp8_blockwise_scaled_mm(a.data_ptr(), lda, b.data_ptr(), ldb, sa_p, sa.stride(0), sa.stride(1), sb_p, sb.stride(0),
                                              sb.stride(1), out.data_ptr(), n, dtype_code(dtype), m, n, k, scratch.partial, scratch.partial_bytes,
                                              here.stream);
    }
    return rc == 0 ? THPVariable_Wrap(std::move(out)) : none();
  });
}

// rowcol_mm(a, b, scales_a, scales_b, out_dtype, bias | None, is_int8, dispatched) -> [M, N]
PyObject* rowcol_mm(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 8) return PyErr_Format(PyExc_TypeError, "rowcol_mm takes 8 arguments");
  return guarded([&]() -> PyObject* {
    const Tensor *ap = gpu_tensor(args[0]), *bp = gpu_tensor(args[1]), *sap = gpu_tensor(args[2]), *sbp = gpu_tensor(args[3]), *bias;
    at::ScalarType dtype;
    if (!ap || !bp || !sap || !sbp || !optional_tensor(args[5], bias) || !out_dtype_of(args[4], dtype)) return none();
    const bool int8 = args[6] == Py_True;
    const Tensor &a = *ap, &b = *bp, &sa = *sap, &sb = *sbp;
    if (!bound || (args[7] != Py_True && (!direct(a, b, sa, sb) || !plain(bias)))) return none();
    if (!mm_operands(a, b, int8 ? at::kChar : FP8)) return none();
    const int64_t m = a.size(0), k = a.size(1), n = b.size(1);
    if (sa.scalar_type() != at::kFloat || sb.scalar_type() != at::kFloat || sa.numel() != m || sb.numel() != n) return none();
    if (!sa.is_contiguous() || !sb.is_contiguous() || sa.device() != a.device() || sb.device() != a.device()) return none();
    if (!bias_fits(bias, n, dtype, a)) return none();
    Tensor out;
    int rc;
    {
      ReleaseGil unlocked;
      Launch here(a.device());
      out = empty({m, n}, dtype, here.device);
      Scratch scratch(here.device, here.stream, 0, m, n, k);
      rc = (int8 ? lib.sglq_int8_scaled_mm : lib.sglq_fp8_scaled_mm)(
          a.data_ptr(), m > 1 ? a.stride(0) : k, b.data_ptr(), n > 1 ? b.stride(1) : k, static_cast<const float*>(sa.data_ptr()),
          static_cast<const float*>(sb.data_ptr()), bias ? bias->data_ptr() : nullptr, out.data_ptr(), n, dtype_code(dtype), m, n, k,
          scratch.partial, scratch.partial_bytes, here.stream);
    }
    return rc == 0 ? THPVariable_Wrap(std::move(out)) : none();
  });
}

inline PyObject* pair_of(Tensor a, Tensor b) {
  PyObject* first = THPVariable_Wrap(std::move(a));
  if (!first) return nullptr;
  PyObject* second = THPVariable_Wrap(std::move(b));
  PyObject* t = second ? PyTuple_New(2) : nullptr;
  if (!t) {
    Py_DECREF(first);
    Py_XDECREF(second);
    return nullptr;
  }
  PyTuple_SET_ITEM(t, 0, first);
  PyTuple_SET_ITEM(t, 1, second);
  return t;
}

// group_quant_fp8(x, group_size, eps, column_major_scales, padded) -> (codes, scales): the buffers of
// sglang_per_token_group_quant_fp8 in its fp32 layouts; column-major scales for 2-D inputs.
PyObject* group_quant_fp8(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 5) return PyErr_Format(PyExc_TypeError, "group_quant_fp8 takes 5 arguments");
  return guarded([&]() -> PyObject* {
    const Tensor* xp = gpu_tensor(args[0]);
    if (!xp || !direct(*xp)) return none();
    const Tensor& x = *xp;
    const long group = PyLong_AsLong(args[1]);
    const float eps = (float)PyFloat_AsDouble(args[2]);
    if (PyErr_Occurred()) return nullptr;
    const bool column = PyObject_IsTrue(args[3]) == 1, padded = PyObject_IsTrue(args[4]) == 1;
    const int code = dtype_code(x.scalar_type());
    if (code < 0 || x.dim() != 2 || !x.is_contiguous() || x.numel() == 0 || group <= 0 || x.size(1) % group != 0) return none();
    const int64_t m = x.size(0), k = x.size(1), g = k / group;
    Tensor q, s;
    int rc;
    {
      ReleaseGil unlocked;
      Launch here(x.device());
      q = empty({m, k}, FP8, here.device);
      if (column) {
        const int64_t rows = padded ? (m + 3) / 4 * 4 : m;
        s = empty({g, rows}, at::kFloat, here.device);
        const int64_t sizes[2] = {m, g}, strides[2] = {1, rows};
        s.unsafeGetTensorImpl()->set_sizes_and_strides(at::IntArrayRef(sizes, 2), at::IntArrayRef(strides, 2));
      } else {
        s = empty({m, g}, at::kFloat, here.device);
      }
      rc = lib.sglq_per_token_group_quant_fp8(x.data_ptr(), code, q.data_ptr(), static_cast<float*>(s.data_ptr()), m, k, (int)group, s.stride(0),
                                              s.stride(1), eps, -448.0f, 448.0f, here.stream);
    }
    return rc == 0 ? pair_of(std::move(q), std::move(s)) : none();
  });
}

// token_quant(x, is_int8) -> (codes, scales [..., 1])
PyObject* token_quant(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 2) return PyErr_Format(PyExc_TypeError, "token_quant takes 2 arguments");
  return guarded([&]() -> PyObject* {
    const Tensor* xp = gpu_tensor(args[0]);
    if (!xp || !direct(*xp)) return none();
    const Tensor& x = *xp;
    const bool int8 = args[1] == Py_True;
    const int code = dtype_code(x.scalar_type());
    if (code < 0 || x.dim() < 1 || (!int8 && x.dim() != 2) || !x.is_contiguous() || x.numel() == 0) return none();
    const int64_t k = x.size(-1), m = x.numel() / k;
    if (!int8 && k % 8 != 0) return none();
    Tensor q, s;
    int rc;
    {
      ReleaseGil unlocked;
      Launch here(x.device());
      q = empty(x.sizes(), int8 ? at::kChar : FP8, here.device);
      s = empty(output_shape(x, 1), at::kFloat, here.device);
      float* s_p = static_cast<float*>(s.data_ptr());
      rc = int8 ? lib.sglq_per_token_quant_int8(x.data_ptr(), code, q.data_ptr(), s_p, nullptr, m, k, here.stream)
                : lib.sglq_per_token_quant_fp8(x.data_ptr(), code, q.data_ptr(), s_p, m, k, here.stream);
    }
    return rc == 0 ? pair_of(std::move(q), std::move(s)) : none();
  });
}

// ---------------------------------------------------------------------------
// experts(a, w1_q, w2_q, w1_scale, w2_scale, topk_weights, topk_ids, expert_offsets, problem_sizes1,
// problem_sizes2) -> [m, k]: cutlass_fused_experts_fp8 (moe/cutlass_moe.py) as four to six launches where the tables
// fit one launch (prepare and quantize, together on few slots; GEMM, SiLU and quantize, one launch on 256-, 32- and 64-row tiles where that is faster; GEMM; combine) from twelve, and
// one allocation beside the result's from eleven: a layer of a few tokens was bound by about 95 us of host
// time around 30-50 us of GPU work.
// ---------------------------------------------------------------------------
inline bool int32_buffer(const Tensor& t, int64_t count, const Tensor& like) {
  return t.scalar_type() == at::kInt && t.is_contiguous() && t.numel() >= count && t.device() == like.device();
}
inline bool expert_weight(const Tensor& w, int64_t e, int64_t k, int64_t n, const Tensor& scale, const Tensor& like) {
  return w.dim() == 3 && w.scalar_type() == FP8 && w.size(0) == e && w.size(1) == k && w.size(2) == n && w.stride(1) == 1 &&
         w.stride(2) % 16 == 0 && w.stride(2) >= k && w.stride(0) % 16 == 0 && aligned(w, 16) && w.device() == like.device() &&
         scale.dim() == 3 && scale.scalar_type() == at::kFloat && scale.size(0) == e && scale.size(1) == (k + 127) / 128 &&
         scale.size(2) == (n + 127) / 128 && scale.device() == like.device();
}

PyObject* experts(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 10) return PyErr_Format(PyExc_TypeError, "experts takes 10 arguments");
  return guarded([&]() -> PyObject* {
    const Tensor* t[10];
    for (int i = 0; i < 10; ++i) {
      t[i] = gpu_tensor(args[i]);
      if (!t[i]) return none();
    }
    const Tensor &x = *t[0], &w1 = *t[1], &w2 = *t[2], &s1 = *t[3], &s2 = *t[4], &weights = *t[5], &ids = *t[6], &offsets = *t[7],
                 &sizes1 = *t[8], &sizes2 = *t[9];
    if (!direct(x, w1, w2, s1, s2, weights)) return none();
    if (!activations(x) || x.dim() != 2 || w1.dim() != 3 || w2.dim() != 3 || ids.dim() != 2 || weights.dim() != 2) return none();
    const int64_t m = x.size(0), k = x.size(1), e = w1.size(0), n = w2.size(1), topk = ids.size(1), rows = m * topk;
    if (e == 0 || n == 0 || topk == 0 || k % 128 != 0 || n % 128 != 0 || ids.size(0) != m || rows >= (int64_t(1) << 31)) return none();
    if (!expert_weight(w1, e, k, 2 * n, s1, x) || !expert_weight(w2, e, n, k, s2, x)) return none();
    const bool float_weights = weights.scalar_type() == at::kFloat;
    if ((!float_weights && weights.scalar_type() != x.scalar_type()) || !weights.is_contiguous() || weights.size(0) != m ||
        weights.size(1) != topk || weights.device() != x.device())
      return none();
    if (!int32_buffer(ids, rows, x) || !int32_buffer(offsets, e + 1, x) || !int32_buffer(sizes1, 3 * e, x) || !int32_buffer(sizes2, 3 * e, x))
      return none();
    const int code = dtype_code(x.scalar_type());
    const bool one_block = rows <= 32768 && e <= 512;
    const int64_t layer_rows = one_block ? lib.sglq_grouped_layer_rows(e, m, topk, n, k) : 0;
    const bool walked = layer_rows == 256, tiled = layer_rows != 0 && !walked;
    const int64_t plan_rows = layer_rows ? layer_rows : lib.sglq_grouped_plan_rows(e, rows, k);
    const int64_t plan_rows2 = layer_rows ? layer_rows : lib.sglq_grouped_plan_rows(e, rows, n);
    const bool shared_plan = plan_rows == plan_rows2;  // (written by the tables, or by the first GEMM: a launch of 5 us less on 48000 slots, 2210 us a layer)
    // GEMM 1 gathers its rows from the tokens' codes, written once.  Quantization + GEMM 1, without and with (us), tokens x experts x
    // top-k, hidden x intermediate: 2500 x 32 x 8, 7168 x 2048 664 -> 626; 600 x 32 x 8 239 -> 223; 2500 x 16 x 3 266 -> 255;
    // 3000 x 16 x 4, 4096 x 1408 194.5 -> 187.8; on 6000 x 16, 2048 x 768 top-8 186 -> 173, top-3 78.5 and 78.4, top-2 68.0 -> 71.4:
    // two copies of the codes cost less than the gathering.
    const bool gathers = topk > 2 && (walked || (!tiled && lib.sglq_grouped_gathers(e, rows, k) != 0));
    // Few slots: the quantization runs beside the tables, in their launch (a launch of 5 us less; its blocks find their rows from all the ids).  Layers without and with
    // (us), tokens x experts x top-k, hidden x intermediate: 1 x 64 x 6, 2048 x 1408 32.3 -> 28.7; 8 x 128 x 8, 2048 x 768 46.9 -> 43.1; 8 x 32 x 8, 7168 x 2048 223.8 -> 220.5; at 2048 slots
    // 256 x 128 x 8 144.0 -> 140.0, 512 x 16 x 4, 5120 x 1536 136.6 -> 134.7, but 1024 x 8 x 2, 6144 x 2048, two blocks a CU, 158.3 -> 159.4.
    const bool joins = rows <= 2048 && m <= 512 && e <= 512 && topk <= 64;
    const int64_t plan_bytes = round256(16 * (rows / 16 + e + 1));
    // On 256-row tiles the tables come with both GEMMs' walks, and GEMM 1 with the activation and its quantization behind it.  Up to 128 rows an expert
    // always, above from 96 tiles on (3/8 of the 256 CUs, on which this was measured): a tile's rows take it up to 8 us, a launch of its own 2.5 us and its bytes (GEMM 1 and the activation's launch -> one launch, us:
    // 2500 tokens x 32 experts x 8, 7168 x 2048 582 -> 570; 777 tokens 267 -> 252; 2048 x 64 x 8, 4096 x 1024 211 -> 191; 1500 x 8 x 3, 1024 x 640 24.2 -> 20.0; of 40 layers of 20 to 128 rows
    // an expert 0.944 on average, 1.013 at most; on few tiles of more rows 881 x 5 x 2, 3200 x 384 37.1 -> 38.5, 606 x 8 x 3, 3072 x 1024 37.2 -> 38.4).
    int64_t walk2_at = 0;
    const int64_t walk_bytes = walked ? lib.sglq_grouped_walk_bytes(e, rows, n, k, &walk2_at) : 0;
    // ... and on 32- and 64-row tiles, by their number (a launch less, 3 to 17 us of 35 to 280)
    const bool activates_few = one_block && !walked && !gathers && plan_rows <= 64 && lib.sglq_grouped_few_rows_activates(e, m, topk, n, k, plan_rows) != 0;
    const bool activates = walked && (rows < 129 * e || (rows / 256 + e / 2) * (n / 128) >= 96), maps_rows = walked || gathers || !one_block;
    // expert-major rows: quantized activations (dead once GEMM 1 has run) under GEMM 2's output, GEMM 1's
    // output, the quantized intermediate
    const int64_t codes1 = round256(rows * k), scales1 = round256(rows * (k / 128) * 4), c2 = round256(rows * k * 2);
    const int64_t c1 = activates || activates_few ? 0 : round256(rows * 2 * n * 2), codes2 = round256(rows * n), scales2 = round256(rows * (n / 128) * 4);
    const int64_t head = codes1 + scales1 > c2 ? codes1 + scales1 : c2, map = round256(rows * 4);
    Tensor out;
    int rc;
    {
      ReleaseGil unlocked;
      Launch here(x.device());
      out = empty({m, k}, x.scalar_type(), here.device);
      Tensor arena = empty({head + c1 + codes2 + scales2 + plan_bytes + map + (maps_rows ? map : 0) + walk_bytes}, at::kByte, here.device);
      char* base = static_cast<char*>(arena.data_ptr());
      char *q1 = base, *y1 = base + head, *q2 = y1 + c1, *plan = q2 + codes2 + scales2;
      float *f1 = reinterpret_cast<float*>(q1 + codes1), *f2 = reinterpret_cast<float*>(q2 + codes2);
      int32_t *slot_map = reinterpret_cast<int32_t*>(plan + plan_bytes), *row_map = reinterpret_cast<int32_t*>(plan + plan_bytes + map);
      const int32_t* ids_p = static_cast<const int32_t*>(ids.data_ptr());
      int32_t *off_p = static_cast<int32_t*>(offsets.data_ptr()), *ps1 = static_cast<int32_t*>(sizes1.data_ptr()),
              *ps2 = static_cast<int32_t*>(sizes2.data_ptr());
      char* const walk1 = reinterpret_cast<char*>(row_map) + map;
      char* const walk2 = walk1 + walk2_at;
      if (joins) {
        rc = lib.sglq_prepare_moe_layer_quant(ids_p, off_p, ps1, ps2, slot_map, walked || gathers ? row_map : nullptr, topk, rows, e, n, k, plan_rows,
                                              rows / plan_rows + e, plan, walked ? walk1 : nullptr, walk_bytes, x.data_ptr(), code, q1, f1, gathers, 1e-10f,
                                              here.stream);
      } else if (walked) {
        rc = lib.sglq_prepare_moe_layer_walks(ids_p, off_p, ps1, ps2, slot_map, row_map, topk, rows, e, n, k, plan, walk1, walk_bytes, here.stream);
      } else if (one_block && gathers) {
        rc = lib.sglq_prepare_moe_layer_rows(ids_p, off_p, ps1, ps2, slot_map, row_map, topk, rows, e, n, k, plan_rows, rows / plan_rows + e, plan,
                                             here.stream);
      } else if (one_block) {
        rc = lib.sglq_prepare_moe_layer(ids_p, off_p, ps1, ps2, slot_map, rows, e, n, k, plan_rows, rows / plan_rows + e, plan, here.stream);
      } else {
        at::NoGradGuard no_grad;
        arena.narrow(0, reinterpret_cast<char*>(slot_map) - base, rows * 4).fill_(255);  // -1: slots routed to nobody
        rc = lib.sglq_prepare_moe_input(ids_p, off_p, nullptr, ps1, ps2, row_map, slot_map, rows, topk, e, n, k, here.stream);
      }
      auto grouped = [&](const void* q, const float* f, const Tensor& w, const Tensor& s, void* y, const int32_t* sizes, int64_t depth,
                         int64_t width, int64_t tile_rows, bool planned, const char* walk, const int32_t* map_p) {
        const float* s_p = static_cast<const float*>(s.data_ptr());
        const int64_t ldb = w.stride(2), bs = e > 1 ? w.stride(0) : width * depth;
        if (walked)
          return lib.sglq_fp8_blockwise_scaled_grouped_mm_walked(q, depth, map_p ? m : rows, map_p, w.data_ptr(), ldb, bs, f, 1, rows, s_p, s.stride(0),
                                                                 s.stride(1), s.stride(2), y, width, code, e, rows, width, depth, plan, plan_bytes,
                                                                 walk, here.stream);
        if (tiled)
          return lib.sglq_fp8_blockwise_scaled_grouped_mm_tiled(q, depth, w.data_ptr(), ldb, bs, f, 1, rows, s_p, s.stride(0), s.stride(1), s.stride(2), y,
                                                                width, code, tile_rows, e, rows, width, depth, plan, plan_bytes, here.stream);
        return planned ? lib.sglq_fp8_blockwise_scaled_grouped_mm_planned(q, depth, w.data_ptr(), ldb, bs, f, 1, rows, s_p, s.stride(0),
                                                                          s.stride(1), s.stride(2), y, width, code, tile_rows, e, rows, width,
                                                                          depth, plan, plan_bytes, here.stream)
                       : lib.sglq_fp8_blockwise_scaled_grouped_mm(q, depth, w.data_ptr(), ldb, bs, f, 1, rows, s_p, s.stride(0),
                                                                  s.stride(1), s.stride(2), y, width, code, sizes, off_p, e, rows, width, depth,
                                                                  plan, plan_bytes, here.stream);
      };
      if (gathers) {
        if (rc == 0 && !joins)
          rc = lib.sglq_per_token_group_quant_fp8_scatter_scales_cm(x.data_ptr(), code, q1, f1, slot_map, m, k, topk, rows, 1e-10f, here.stream);
        if (rc == 0 && walked && !activates) rc = grouped(q1, f1, w1, s1, y1, ps1, k, 2 * n, plan_rows, true, walk1, row_map);
        else if (rc == 0 && !walked)
          rc = lib.sglq_fp8_blockwise_scaled_grouped_mm_gathered(q1, k, m, row_map, w1.data_ptr(), w1.stride(2), e > 1 ? w1.stride(0) : 2 * n * k, f1,
                                                                 1, rows, static_cast<const float*>(s1.data_ptr()), s1.stride(0), s1.stride(1),
                                                                 s1.stride(2), y1, 2 * n, code, ps1, off_p, one_block ? plan_rows : 0, e, rows,
                                                                 2 * n, k, plan, plan_bytes, here.stream);
      } else {
        if (rc == 0 && !joins) rc = lib.sglq_per_token_group_quant_fp8_scatter_cm(x.data_ptr(), code, q1, f1, slot_map, m, k, topk, rows, 1e-10f, here.stream);
        if (rc == 0 && !activates && !activates_few) rc = grouped(q1, f1, w1, s1, y1, ps1, k, 2 * n, plan_rows, one_block, walk1, nullptr);
      }
      if (rc == 0 && activates)
        rc = lib.sglq_fp8_blockwise_scaled_grouped_mm_silu(q1, k, gathers ? m : rows, gathers ? row_map : nullptr, w1.data_ptr(), w1.stride(2),
                                                           e > 1 ? w1.stride(0) : 2 * n * k, f1, 1, rows, static_cast<const float*>(s1.data_ptr()),
                                                           s1.stride(0), s1.stride(1), s1.stride(2), q2, f2, code, 1e-10f, e, rows, 2 * n, k, plan,
                                                           plan_bytes, walk1, here.stream);
      else if (rc == 0 && activates_few)
        rc = lib.sglq_fp8_blockwise_scaled_grouped_mm_silu_few_rows(q1, k, w1.data_ptr(), w1.stride(2), e > 1 ? w1.stride(0) : 2 * n * k, f1, 1, rows,
                                                              static_cast<const float*>(s1.data_ptr()), s1.stride(0), s1.stride(1), s1.stride(2), q2, f2,
                                                              code, 1e-10f, e, rows, 2 * n, k, plan, plan_bytes, plan_rows, here.stream);
      else if (rc == 0) rc = lib.sglq_silu_and_mul_group_quant_fp8_cm(y1, code, q2, f2, rows, n, 1e-10f, here.stream);
      if (rc == 0) rc = grouped(q2, f2, w2, s2, base, ps2, n, k, plan_rows2, shared_plan, walk2, nullptr);
      if (rc == 0 && float_weights)
        rc = lib.sglq_apply_shuffle_mul_sum_f32(base, out.data_ptr(), slot_map, static_cast<const float*>(weights.data_ptr()), code, m, topk, k,
                                                rows, here.stream);
      else if (rc == 0)
        rc = lib.sglq_apply_shuffle_mul_sum(base, out.data_ptr(), slot_map, weights.data_ptr(), code, m, topk, k, rows, here.stream);
    }
    return rc == 0 ? THPVariable_Wrap(std::move(out)) : none();
  });
}

// ---------------------------------------------------------------------------
// bind({name: address}); kept_scratch(device index); release_workspaces()
// ---------------------------------------------------------------------------
PyObject* bind(PyObject*, PyObject* table) {
  EntryPoints e;
#define X(name)                                                                                                  \
  {                                                                                                              \
    PyObject* v = PyDict_Check(table) ? PyDict_GetItemString(table, #name) : nullptr;                            \
    if (!v) return PyErr_Format(PyExc_KeyError, "bind: the address of %s is missing", #name);                    \
    e.name = reinterpret_cast<decltype(e.name)>(PyLong_AsVoidPtr(v));                                            \
    if (!e.name) return PyErr_Occurred() ? nullptr : PyErr_Format(PyExc_ValueError, "bind: %s is null", #name);  \
  }
  SGLQ_HOST_ENTRY_POINTS(X)
#undef X
  lib = e;
  bound = true;
  return none();
}

PyObject* entry_points(PyObject*, PyObject*) {
  PyObject* names = PyList_New(0);
  if (!names) return nullptr;
#define X(name)                                             \
  {                                                         \
    PyObject* s = PyUnicode_FromString(#name);              \
    if (!s || PyList_Append(names, s) < 0) {                \
      Py_XDECREF(s);                                        \
      Py_DECREF(names);                                     \
      return nullptr;                                       \
    }                                                       \
    Py_DECREF(s);                                           \
  }
  SGLQ_HOST_ENTRY_POINTS(X)
#undef X
  return names;
}

// (address, bytes) of the buffer that eager calls on the device's current stream keep
PyObject* kept_scratch(PyObject*, PyObject* index) {
  return guarded([&]() -> PyObject* {
    const long i = PyLong_AsLong(index);
    if (i == -1 && PyErr_Occurred()) return nullptr;
    Launch here(c10::Device(c10::kCUDA, static_cast<c10::DeviceIndex>(i)));
    auto w = workspace_of(here.device, here.stream);
    return Py_BuildValue("NL", PyLong_FromVoidPtr(w->base), static_cast<long long>(CODES_BYTES + SPLITK_BYTES));
  });
}

PyObject* release_workspaces(PyObject*, PyObject*) {
  return guarded([&]() -> PyObject* {
    Workspaces old;
    {
      std::lock_guard<std::mutex> guard(workspaces_lock);
      old.swap(workspaces);
    }
    return none();
  });
}

#define FAST(f) reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)), METH_FASTCALL
PyMethodDef methods[] = {
    {"bind", bind, METH_O, "bind({name: address}) of the library's entry points"},
    {"entry_points", entry_points, METH_NOARGS, "the names that bind() wants"},
    {"kept_scratch", kept_scratch, METH_O, "(address, bytes) of the scratch kept for the device's current stream"},
    {"release_workspaces", release_workspaces, METH_NOARGS, "give the kept scratch buffers back to torch's allocator"},
    {"pow2_scales_known", pow2_scales_known, METH_O, "whether note_pow2_scales has been given this tensor as it is now"},
    {"note_pow2_scales", note_pow2_scales, METH_O, "remember that a weight's block scales are powers of two"},
    {"block_linear", FAST(block_linear), "quantize and multiply with a block-scaled weight, or None"},
    {"token_linear", FAST(token_linear), "quantize per token and multiply with a per-channel-scaled weight, or None"},
    {"blockwise_mm", FAST(blockwise_mm), "block-scaled FP8 GEMM, or None"},
    {"rowcol_mm", FAST(rowcol_mm), "per-token / per-channel-scaled GEMM, or None"},
    {"group_quant_fp8", FAST(group_quant_fp8), "per-token-group FP8 quantization, or None"},
    {"token_quant", FAST(token_quant), "per-token quantization, or None"},
    {"experts", FAST(experts), "an expert layer, or None"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", "Host path of the per-layer operators", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) { return PyModule_Create(&module); }
