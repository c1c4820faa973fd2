// The operators' way from torch to the kernels, in native code: torch.ops.xla.quantized_matmul and
// torch.ops.xla_amd.weight_only_tiled on ROCm tensors check their arguments, allocate their result (and workspace),
// and call the C entry points of libxla_amd_qmm.so.  Through Python and ctypes that took 17 - 19 us per eager call,
// longer than the kernels of a decode step (5 - 12 us each).
//
// Only the ordinary call is handled here.  Whatever needs more - a weight without its tiled copy yet, arguments that
// will be refused (the messages are Python's), empty tensors, strided weights - goes to the Python formulation of the
// same operator (xla_amd::quantized_matmul_general, xla_amd::weight_only_tiled_general), which accepts and refuses
// exactly the same calls.
#include <ATen/core/dispatch/Dispatcher.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <ATen/ops/empty.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/Event.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <torch/library.h>

#include <algorithm>
#include <atomic>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <optional>
#include <unordered_map>
#include <vector>

#include "xla_amd_qmm.h"

namespace {

using at::Tensor;
typedef std::optional<Tensor> OptTensor;

// Dispatch decisions since the library was loaded, in the order of the Python module's `counters` (whose last, the copies
// made, happen in Python only).
enum Counter { kSkinny, kWoGemm, kGeneric, kW8a8, kW8a8Generic, kPackHit, kCounters };
std::atomic<int64_t> g_counters[kCounters];
void count(Counter c) { g_counters[c].fetch_add(1, std::memory_order_relaxed); }

int dt_of(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return XLA_AMD_DT_F32;
    case at::kBFloat16: return XLA_AMD_DT_BF16;
    case at::kHalf: return XLA_AMD_DT_F16;
    default: return -1;
  }
}
at::ScalarType type_of(int dt) {
  return dt == XLA_AMD_DT_F32 ? at::kFloat : dt == XLA_AMD_DT_BF16 ? at::kBFloat16 : at::kHalf;
}
int promote(int a, int b) { return a == b ? a : XLA_AMD_DT_F32; }

void check(int rc, const char* what) {
  TORCH_CHECK(rc == XLA_AMD_QMM_OK, what, " failed (code ", rc, "): ", xla_amd_qmm_last_error());
}

// ---- tiled copies of weights passed to the operator -------------------------------------------------------------
// A mirror of the Python module's cache, which makes the copies and says when they are to be dropped.  An entry holds
// its weight weakly: the address of its TensorImpl cannot be taken by another tensor while the entry exists.  It
// stands as long as the weight is unmodified (version counter, storage address).
// The copy is made by a kernel on the stream of whichever call came first and read on the stream of any later one, so
// an entry keeps that stream and an event behind the kernel.
struct Copy {
  c10::weak_intrusive_ptr<c10::TensorImpl> weight;
  int64_t version;
  const void* data;
  int64_t bits;
  Tensor tiled;
  c10::Stream made_on;
  c10::Event made;                   // recorded behind the kernel that makes the copy
  bool complete;                     // that kernel has been seen to be done
  std::vector<c10::Stream> used_on;  // other streams the allocator knows to read the copy
};
struct Cache {
  std::mutex mu;
  std::unordered_map<const c10::TensorImpl*, Copy> of;
};
Cache& cache() {
  static Cache* c = new Cache;  // (never destroyed: its tensors would outlive the allocator)
  return *c;
}
c10::Stream current_stream(const Tensor& t) {
  return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).unwrap();
}
int64_t version_of(const Tensor& w) { return w.is_inference() ? -1 : (int64_t)w._version(); }

int64_t remember_tiled(const Tensor& w, int64_t bits, const Tensor& tiled) {
  c10::TensorImpl* const key = w.unsafeGetTensorImpl();
  const c10::Stream made_on = current_stream(tiled);
  Copy copy{c10::weak_intrusive_ptr<c10::TensorImpl>(w.getIntrusivePtr()), version_of(w), w.data_ptr(), bits, tiled, made_on,
            c10::Event(made_on.device_type()), false, {}};
  copy.made.record(made_on);
  std::lock_guard<std::mutex> lock(cache().mu);
  cache().of.insert_or_assign(key, std::move(copy));
  return (int64_t)(uintptr_t)key;
}
void forget_tiled(int64_t key) {
  std::optional<Copy> gone;  // (destroyed after the lock is released)
  std::lock_guard<std::mutex> lock(cache().mu);
  auto it = cache().of.find((const c10::TensorImpl*)(uintptr_t)key);
  if (it == cache().of.end()) return;
  gone.emplace(std::move(it->second));
  cache().of.erase(it);
}
// Makes the copy safe to read by work that is launched on the current stream from here on, and keeps its memory from
// being handed out again before that work is done.  (The lock is held.)
void use_on_current_stream(Copy& c) {
  if (c.complete && c10::hip::getCurrentHIPStream(c.made_on.device_index()).id() == c.made_on.id()) return;  // the usual case
  const c10::Stream now = current_stream(c.tiled);
  if (!c.complete) {
    // (event queries and waits are refused while any thread captures, unless this thread's capture mode is relaxed)
    c10::hip::HIPStreamCaptureModeGuard relaxed(hipStreamCaptureModeRelaxed);
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    if (c.made.query()) {
      c.complete = true;
    } else {
      C10_HIP_CHECK(hipStreamIsCapturing(c10::hip::getCurrentHIPStream(now.device_index()), &capturing));
      if (capturing != hipStreamCaptureStatusNone) {
        // the graph may be replayed on any stream, and cannot wait for work outside of it: wait for it here
        c.made.synchronize();
        c.complete = true;
      } else if (now != c.made_on) {
        c.made.block(now);
      }
    }
  }
  if (now != c.made_on && std::find(c.used_on.begin(), c.used_on.end(), now) == c.used_on.end()) {
    c.tiled.record_stream(now);
    c.used_on.push_back(now);
  }
}
Tensor find_tiled(const Tensor& w, int64_t bits) {
  std::lock_guard<std::mutex> lock(cache().mu);
  auto it = cache().of.find(w.unsafeGetTensorImpl());
  if (it == cache().of.end()) return Tensor();
  Copy& c = it->second;
  if (c.bits != bits || c.data != w.data_ptr() || c.version != version_of(w)) return Tensor();
  use_on_current_stream(c);
  count(kPackHit);
  return c.tiled;
}
// The same for a copy that Python has found in its own cache; false if it is no longer the one recorded under its key.
bool use_tiled(int64_t key, const Tensor& tiled) {
  std::lock_guard<std::mutex> lock(cache().mu);
  auto it = cache().of.find((const c10::TensorImpl*)(uintptr_t)key);
  if (it == cache().of.end() || !it->second.tiled.is_same(tiled)) return false;
  use_on_current_stream(it->second);
  return true;
}

// ---- one call ---------------------------------------------------------------------------------------------------

void* stream_of(const Tensor& t) {
  return (void*)c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream();
}
const void* ptr(const OptTensor& t) { return t ? t->data_ptr() : nullptr; }

Tensor empty_like_rows(const Tensor& x, int64_t n, int dt) {
  auto sizes = x.sizes().vec();
  sizes.back() = n;
  return at::empty(sizes, x.options().dtype(type_of(dt)));
}
Tensor workspace(const Tensor& x, size_t bytes) { return at::empty({(int64_t)bytes}, x.options().dtype(at::kByte)); }

// x [..., k] with at least one row, scale and zero point on x's device in supported dtypes
bool ordinary(const Tensor& x, const Tensor& scale, const OptTensor& zp) {
  return x.dim() >= 1 && x.numel() > 0 && dt_of(x.scalar_type()) >= 0 && dt_of(scale.scalar_type()) >= 0 &&
         scale.device() == x.device() && scale.numel() > 0 &&
         (!zp || (dt_of(zp->scalar_type()) >= 0 && zp->device() == x.device() && zp->numel() > 0));
}

// The weight-only product against the tiled copy `tiled`, or against `w` in the operator's layout (XLA_AMD_W_*) where
// the shape runs the generic kernel.  No value: not an ordinary call.
std::optional<Tensor> weight_only(const Tensor& x_in, const Tensor& tiled, const Tensor* w, int layout, int64_t n,
                                  int64_t k, int64_t c, int bits, const Tensor& scale_in, const OptTensor& zp_in) {
  const int64_t m = x_in.numel() / k;
  const int x_dt = dt_of(x_in.scalar_type()), s_dt = dt_of(scale_in.scalar_type());
  const int zp_dt = zp_in ? dt_of(zp_in->scalar_type()) : x_dt;
  const int out_dt = promote(x_dt, s_dt);
  if (c != k && (s_dt != x_dt || zp_dt != x_dt)) return std::nullopt;
  int kern = xla_amd_qmm_dispatch(m, n, k, c, bits, x_dt, 0);
  // (the tiled GEMM for blockwise / int4 weights computes in one dtype throughout)
  if (kern == XLA_AMD_KERNEL_WEIGHT_ONLY_GEMM && (c != k || bits == 4) && m > 32 && (s_dt != x_dt || zp_dt != x_dt))
    kern = XLA_AMD_KERNEL_SKINNY_MFMA;
  if (kern == XLA_AMD_KERNEL_WEIGHT_ONLY_GEMM || kern == XLA_AMD_KERNEL_SKINNY_MFMA) {
    if (!tiled.defined()) return std::nullopt;
  } else if (!w || !w->is_contiguous()) {
    return std::nullopt;
  }
  const c10::DeviceGuard guard(x_in.device());
  const Tensor x = x_in.contiguous(), scale = scale_in.contiguous();
  const OptTensor zp = zp_in ? OptTensor(zp_in->contiguous()) : std::nullopt;
  Tensor out = empty_like_rows(x, n, out_dt);
  void* const stream = stream_of(x);
  if (kern == XLA_AMD_KERNEL_WEIGHT_ONLY_GEMM && x_dt == XLA_AMD_DT_F32) {
    count(kWoGemm);
    const size_t bytes = xla_amd_qmm_weight_only_gemm_f32_workspace_bytes(m, n, k);
    const Tensor ws = bytes ? workspace(x, bytes) : Tensor();
    check(xla_amd_qmm_weight_only_gemm_f32((const float*)x.data_ptr(), tiled.data_ptr(), scale.data_ptr(), ptr(zp),
                                           (float*)out.data_ptr(), bytes ? ws.data_ptr() : nullptr, bytes, m, n, k, s_dt,
                                           zp_dt, stream),
          "weight_only_gemm_f32");
  } else if (kern == XLA_AMD_KERNEL_WEIGHT_ONLY_GEMM) {
    count(kWoGemm);
    const size_t bytes = xla_amd_qmm_weight_only_gemm_workspace_bytes(m, n, k, c, bits);
    const Tensor ws = bytes ? workspace(x, bytes) : Tensor();
    check(xla_amd_qmm_weight_only_gemm(x.data_ptr(), tiled.data_ptr(), scale.data_ptr(), ptr(zp), out.data_ptr(),
                                       bytes ? ws.data_ptr() : nullptr, bytes, m, n, k, c, bits, x_dt, s_dt, zp_dt,
                                       x_dt, out_dt, out_dt, stream),
          "weight_only_gemm");
  } else if (kern == XLA_AMD_KERNEL_SKINNY_MFMA) {
    count(kSkinny);
    check(xla_amd_qmm_weight_only_skinny(x.data_ptr(), tiled.data_ptr(), scale.data_ptr(), ptr(zp), out.data_ptr(), m, n,
                                         k, c, bits, x_dt, s_dt, zp_dt, x_dt, out_dt, out_dt, stream),
          "weight_only_skinny");
  } else {
    count(kGeneric);
    check(xla_amd_qmm_weight_only_generic(x.data_ptr(), (const int8_t*)w->data_ptr(), scale.data_ptr(), ptr(zp),
                                          out.data_ptr(), m, n, k, c, layout, x_dt, s_dt, zp_dt, x_dt, out_dt, out_dt, stream),
          "weight_only_generic");
  }
  return out;
}

// Per-token quantization of x and the int8 GEMM.  No value: not an ordinary call.
std::optional<Tensor> w8a8(const Tensor& x_in, const Tensor& w, int64_t n, int64_t k, const Tensor& scale_in,
                           const OptTensor& zp_in) {
  const char* const overflow = std::getenv("XLA_AMD_QMM_OVERFLOW");
  int policy = XLA_AMD_OVERFLOW_SATURATE;
  if (overflow && std::strcmp(overflow, "wrap") == 0) policy = XLA_AMD_OVERFLOW_WRAP;
  else if (overflow && std::strcmp(overflow, "saturate") != 0) return std::nullopt;
  if (!w.is_contiguous()) return std::nullopt;
  const int64_t m = x_in.numel() / k;
  const int x_dt = dt_of(x_in.scalar_type()), s_dt = dt_of(scale_in.scalar_type());
  const int out_dt = promote(s_dt, x_dt);
  const c10::DeviceGuard guard(x_in.device());
  const Tensor x = x_in.contiguous(), scale = scale_in.contiguous();
  const OptTensor zp = zp_in ? OptTensor(zp_in->contiguous()) : std::nullopt;
  Tensor out = empty_like_rows(x, n, out_dt);
  const size_t bytes = xla_amd_qmm_w8a8_linear_workspace_bytes(m, n, k);
  Tensor ws = workspace(x, bytes);
  count(xla_amd_qmm_dispatch(m, n, k, k, 8, XLA_AMD_DT_F32, 1) == XLA_AMD_KERNEL_W8A8_MFMA ? kW8a8 : kW8a8Generic);
  check(xla_amd_qmm_w8a8_linear(x.data_ptr(), (const int8_t*)w.data_ptr(), scale.data_ptr(), ptr(zp), out.data_ptr(),
                                ws.data_ptr(), bytes, m, n, k, x_dt, s_dt, zp ? dt_of(zp->scalar_type()) : XLA_AMD_DT_F32,
                                x_dt, s_dt, s_dt, out_dt, policy, 0, 0, stream_of(x)),
        "w8a8_linear");
  return out;
}

// ---- operators --------------------------------------------------------------------------------------------------

Tensor quantized_matmul(const Tensor& x, const Tensor& w, const Tensor& scale, const OptTensor& zp,
                        std::optional<int64_t> block_size, std::optional<bool> int4_weight,
                        std::optional<bool> quantize_activation) {
  const int64_t block = block_size.value_or(-1);
  const bool int4 = int4_weight.value_or(false), act = quantize_activation.value_or(false);
  if (ordinary(x, scale, zp) && w.scalar_type() == at::kChar && w.device() == x.device() && w.numel() > 0) {
    const int64_t k = x.size(-1);
    std::optional<Tensor> out;
    if (block == -1) {
      if (w.dim() == 2 && scale.dim() == 1 && w.size(1) == k && scale.size(0) == w.size(0) &&
          (!zp || zp->sizes() == scale.sizes())) {
        const int64_t n = w.size(0);
        out = act ? w8a8(x, w, n, k, scale, zp)
                  : weight_only(x, find_tiled(w, int4 ? 4 : 8), &w, XLA_AMD_W_NK, n, k, k, int4 ? 4 : 8, scale, zp);
      }
    } else if (!act && block > 0 && w.dim() == 3 && scale.dim() == 2 && w.size(1) == block &&
               w.size(0) * block == k && scale.size(0) == w.size(0) && scale.size(1) == w.size(2) &&
               (!zp || zp->sizes() == scale.sizes())) {
      out = weight_only(x, find_tiled(w, int4 ? 4 : 8), &w, XLA_AMD_W_SCN, w.size(2), k, block, int4 ? 4 : 8, scale, zp);
    }
    if (out) return *out;
  }
  static const auto general = c10::Dispatcher::singleton().findSchemaOrThrow("xla_amd::quantized_matmul_general", "")
      .typed<Tensor(const Tensor&, const Tensor&, const Tensor&, const OptTensor&, int64_t, bool, bool)>();
  return general.call(x, w, scale, zp, block, int4, act);
}

Tensor weight_only_tiled(const Tensor& x, const Tensor& tiled, const Tensor& scale, const OptTensor& zp, int64_t n,
                         int64_t block_size, bool int4_weight) {
  if (ordinary(x, scale, zp) && tiled.device() == x.device() && n > 0) {
    const int64_t k = x.size(-1), c = block_size == -1 ? k : block_size;
    const int bits = int4_weight ? 4 : 8;
    const size_t need = c > 0 ? xla_amd_qmm_tiled_bytes(n, k, c, bits) : 0;
    if (need > 0 && (size_t)tiled.nbytes() == need) {
      const auto out = weight_only(x, tiled, nullptr, XLA_AMD_W_NK, n, k, c, bits, scale, zp);
      if (out) return *out;
    }
  }
  static const auto general = c10::Dispatcher::singleton().findSchemaOrThrow("xla_amd::weight_only_tiled_general", "")
      .typed<Tensor(const Tensor&, const Tensor&, const Tensor&, const OptTensor&, int64_t, int64_t, bool)>();
  return general.call(x, tiled, scale, zp, n, block_size, int4_weight);
}

}  // namespace

TORCH_LIBRARY_IMPL(xla, CUDA, m) { m.impl("quantized_matmul", quantized_matmul); }
TORCH_LIBRARY_IMPL(xla_amd, CUDA, m) { m.impl("weight_only_tiled", weight_only_tiled); }
TORCH_LIBRARY_FRAGMENT(xla_amd, m) {
  m.def("remember_tiled(Tensor w, int bits, Tensor tiled) -> int", remember_tiled);
  m.def("forget_tiled(int key) -> ()", forget_tiled);
  m.def("use_tiled(int key, Tensor tiled) -> bool", use_tiled);
}

extern "C" int64_t xla_amd_torch_counter(int i) {
  return i >= 0 && i < kCounters ? g_counters[i].load(std::memory_order_relaxed) : 0;
}
