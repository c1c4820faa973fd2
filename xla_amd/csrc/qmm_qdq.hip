// Affine quantize / dequantize of whole tensors (per tensor or per channel):
// HBM-bound elementwise kernels for the quantized_decomposed operators that
// sit on either side of a quantized matmul in PT2E flows.
//
// A contiguous tensor is addressed as [outer, channels, inner]; element
// (o, c, i) uses parameter c (channels == 1: per tensor).  The arithmetic is
// torch's decomposition (torch/ao/quantization/fx/_decomposed.py), op by op in
// f32:  q = cast(clamp(rint(f32(x) * inv_scale[c]) + zp[c], qmin, qmax))
// (rint: half to even); NaN maps to 0.
#include "qmm_common.h"

namespace {

__device__ __forceinline__ int qdq_load_q(const void* q, int64_t i, int q_dt) {
  switch (q_dt) {
    case XLA_AMD_QDT_I8: return ((const int8_t*)q)[i];
    case XLA_AMD_QDT_U8: return ((const uint8_t*)q)[i];
    case XLA_AMD_QDT_I16: return ((const int16_t*)q)[i];
    default: return ((const int32_t*)q)[i];
  }
}
__device__ __forceinline__ void qdq_store_q(void* q, int64_t i, int v, int q_dt) {
  switch (q_dt) {
    case XLA_AMD_QDT_I8: ((int8_t*)q)[i] = (int8_t)v; break;
    case XLA_AMD_QDT_U8: ((uint8_t*)q)[i] = (uint8_t)v; break;
    case XLA_AMD_QDT_I16: ((int16_t*)q)[i] = (int16_t)v; break;
    default: ((int32_t*)q)[i] = v; break;
  }
}

__device__ __forceinline__ int quantize_value(float x, float inv_scale, float zp, float qmin, float qmax) {
  float r = rintf(x * inv_scale) + zp;
  r = fminf(fmaxf(r, qmin), qmax);  // NaN -> qmin by fmaxf/fminf; mapped to 0 below
  return (x != x) ? 0 : (int)r;
}

// The parameters of a call as the caller holds them: scale (or its reciprocal) f32, bf16 or f16, zero point int32 or
// int64 or none.  Converting them beforehand took four launches of a few microseconds each around a
// quantize / dequantize pair: 14336 x 4096 bf16 to f32 103.9 us, 75.7 without them and with the streaming stores below
// (470 MB: 6.2 TB/s).
struct QdqParams {
  const void* scale;
  const void* zp;   // null: 0
  int scale_dt, zp64, reciprocal;  // reciprocal: what multiplies x is 1 / scale
};
// A channel's parameters.  They are requested without a conversion, and converted when they are needed: a conversion
// inside the branch on a type waits for its load, and each load would wait for the one before (a bf16 pair over 4096 x 64
// elements 5.8 us, 5.1 so).
struct RawParams {
  uint32_t scale;
  int zp;
};
__device__ __forceinline__ RawParams qdq_request(const QdqParams& p, uint32_t c) {
  RawParams r = {qmm_load_raw(p.scale, c, p.scale_dt), 0};
  if (p.zp) r.zp = ((const int32_t*)p.zp)[(size_t)c << p.zp64];  // (the low half of an int64)
  return r;
}
__device__ __forceinline__ float qdq_factor(const QdqParams& p, float s) { return p.reciprocal ? 1.0f / s : s; }
__device__ __forceinline__ float qdq_scale(const QdqParams& p, const RawParams& r) {
  return qdq_factor(p, qmm_from_raw(r.scale, p.scale_dt));
}
// ... and those of RUN consecutive channels, in 16-byte pieces (at any element's address).
template <int RUN>
struct RawAlong {
  i32x4 scale[RUN / 4], zp[RUN / 2];
  __device__ __forceinline__ void request(const QdqParams& p, uint32_t c) {
    if (p.scale_dt == XLA_AMD_DT_F32) __builtin_memcpy(scale, (const float*)p.scale + c, RUN * 4);
    else __builtin_memcpy(scale, (const uint16_t*)p.scale + c, RUN * 2);
    if (!p.zp) return;
    if (p.zp64) __builtin_memcpy(zp, (const int64_t*)p.zp + c, RUN * 8);
    else __builtin_memcpy(zp, (const int32_t*)p.zp + c, RUN * 4);
  }
  __device__ __forceinline__ float scale_of(const QdqParams& p, int i) const {
    const uint32_t pair = (uint32_t)scale[i / 8][i / 2 % 4];
    return qdq_factor(p, p.scale_dt == XLA_AMD_DT_F32 ? __int_as_float(scale[i / 4][i % 4])
                                                      : qmm_from_raw(i & 1 ? pair >> 16 : pair & 0xffffu, p.scale_dt));
  }
  __device__ __forceinline__ int zp_of(const QdqParams& p, int i) const {
    return !p.zp ? 0 : p.zp64 ? zp[i / 2][i % 2 * 2] : zp[i / 4][i % 4];
  }
};

// How the elements of a tensor [outer, channels, inner] find their channel.  A thread of the vector forms handles U
// runs of consecutive elements: kOne, one channel; kRow, a run lies within a channel (inner a multiple of the run);
// kAlong, inner == 1, a run lies along the channels (channels a multiple of the run).  kAny: element by element.
// What bounds the vector forms is memory alone as long as a run's channel costs few instructions: 32-bit divisions by
// the row length (the 64-bit ones of kAny take over a hundred instructions), none for kOne; in kAlong a thread's runs
// lie below each other, so that it fetches its channels' parameters (and divides for the quantizer's reciprocals) once
// for kDown of them (4096 x 4096 along the last axis, a bf16 pair: 20 us; element by element 67).
enum Form { kOne, kRow, kAlong, kAny };
constexpr int kThreads = 256;
constexpr int kPerBlock = 4096;  // elements per workgroup of kOne and kRow: several runs in flight per thread
constexpr int kDown = 8;         // rows per thread of kAlong
// Workgroups that keep the chip busy: one run per thread rather than fewer workgroups than that (kAlong, where a run then
// fetches its channels' parameters by itself, a few less).
constexpr int kFill = 4096, kFillAlong = 512;
struct QdqShape {
  int64_t total, outer, channels, inner;
};
// Runs per thread: one where more would leave the chip idle (FEW).
template <Form F, int RUN, bool FEW> constexpr int runs_per_thread() { return FEW ? 1 : F == kAlong ? kDown : kPerBlock / (kThreads * RUN); }
// The thread's runs, if it has any: first + u * stride, u < live (1 .. U), and the channel of run u (kAlong: of every one).
template <Form F, int RUN, uint32_t U>
struct Runs {
  uint32_t first, stride, live;
  bool any;
  __device__ __forceinline__ explicit Runs(const QdqShape& sh) {
    if constexpr (F == kAlong) {
      const uint32_t per_row = (uint32_t)(sh.channels / RUN), rows = (uint32_t)sh.outer;
      const uint32_t t = blockIdx.x * kThreads + threadIdx.x, down = t / per_row;
      const uint32_t row = down * U;
      any = row < rows;
      live = min(U, rows - row);
      first = row * per_row + (t - down * per_row);
      stride = per_row;
    } else {
      const uint32_t runs = (uint32_t)(sh.total / RUN);
      first = blockIdx.x * (kThreads * U) + threadIdx.x;
      stride = kThreads;
      any = first < runs;
      live = min(U, (runs - first + kThreads - 1) / kThreads);
    }
  }
  __device__ __forceinline__ uint32_t run(uint32_t u) const { return first + min(u, live - 1) * stride; }  // (the end repeats the last)
  __device__ __forceinline__ uint32_t channel(const QdqShape& sh, uint32_t run) const {
    if constexpr (F == kOne) return 0;
    if constexpr (F == kRow) return (run / (uint32_t)(sh.inner / RUN)) % (uint32_t)sh.channels;
    return run % stride * RUN;
  }
};

// The parameters of a thread's runs: one channel's per run, or (kAlong) those of the channels of all of them.
template <Form F, int RUN, int U>
struct RunParams {
  RawParams of[F == kAlong ? 1 : U];
  RawAlong<RUN> along;
  __device__ __forceinline__ RunParams(const QdqParams& p, const QdqShape& sh, const Runs<F, RUN, U>& at) {
    if constexpr (F == kAlong) {
      along.request(p, at.channel(sh, at.first));
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u) of[u] = qdq_request(p, at.channel(sh, at.run(u)));
    }
  }
};

// kAny: an element's channel (64-bit divisions, over a hundred instructions, only for tensors that need them) and its
// zero point.
__device__ __forceinline__ uint32_t element_channel(const QdqShape& sh, int64_t t) {
  if (sh.total <= 0xffffffffLL) return (uint32_t)t / (uint32_t)sh.inner % (uint32_t)sh.channels;
  return (uint32_t)((t / sh.inner) % sh.channels);
}
__device__ __forceinline__ int element_zp(const QdqParams& p, uint32_t c) {
  if (!p.zp) return 0;
  return ((const int32_t*)p.zp)[(size_t)c << p.zp64];
}

// Quantize; vector forms: runs of 8, 16-byte aligned x, 8-byte aligned q, 1-byte q, total / 8 < 2^32.
// NT: streaming loads of x.
template <int XT, Form F, bool NT, bool FEW>
__global__ void __launch_bounds__(kThreads)
qdq_quantize_kernel(const void* __restrict__ x, void* __restrict__ q, QdqParams p, QdqShape sh, int q_dt, float qmin,
                    float qmax) {
  if constexpr (F != kAny) {
    constexpr int RUN = 8, U = runs_per_thread<F, RUN, FEW>();
    const Runs<F, RUN, U> at(sh);
    if (!at.any) return;
    constexpr int D = XT == XLA_AMD_DT_F32 ? 2 : 1;
    const RunParams<F, RUN, U> par(p, sh, at);
    i32x4 raw[U][D];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const i32x4* const from = (const i32x4*)x + (size_t)at.run(u) * D;
#pragma unroll
      for (int d = 0; d < D; ++d) raw[u][d] = NT ? __builtin_nontemporal_load(from + d) : from[d];
    }
    float isv[RUN], zv[RUN];
    if constexpr (F == kAlong) {
#pragma unroll
      for (int i = 0; i < RUN; ++i) { isv[i] = par.along.scale_of(p, i); zv[i] = (float)par.along.zp_of(p, i); }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t run = at.run(u);
      float is = 0.f, z = 0.f;
      if constexpr (F != kAlong) { is = qdq_scale(p, par.of[u]); z = (float)par.of[u].zp; }
      uint32_t out[2] = {0, 0};
#pragma unroll
      for (int i = 0; i < RUN; ++i) {
        float f;
        if constexpr (XT == XLA_AMD_DT_F32) {
          f = __int_as_float(raw[u][i / 4][i % 4]);
        } else {
          const uint32_t w = (uint32_t)raw[u][0][i / 2];
          f = qmm_from_raw((i & 1) ? (w >> 16) : (w & 0xffffu), XT);
        }
        if constexpr (F == kAlong) { is = isv[i]; z = zv[i]; }
        out[i / 4] |= ((uint32_t)(uint8_t)quantize_value(f, is, z, qmin, qmax)) << (8 * (i % 4));
      }
      *(i32x2*)((uint8_t*)q + (size_t)run * RUN) = i32x2{(int)out[0], (int)out[1]};
    }
  } else {
    const int64_t t = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (t >= sh.total) return;
    const uint32_t c = element_channel(sh, t);
    qdq_store_q(q, t, quantize_value(qmm_load(x, t, XT), qdq_factor(p, qmm_load(p.scale, c, p.scale_dt)), (float)element_zp(p, c), qmin, qmax), q_dt);
  }
}

// int_subtract != 0: out = cast(f32(q - zp[c]) * scale[c])            (per-channel form)
// int_subtract == 0: out = round(round(cast(q) - zp[c]) * scale[c])   (per-tensor form, tensor ops in out's dtype)
__device__ __forceinline__ float dequantize_value(int qv, int z, float sc, int out_dt, int int_subtract) {
  if (int_subtract) return (float)(qv - z) * sc;
  // (zero point and scale are host scalars there: they enter the arithmetic as f32)
  const float a = qmm_round_dt((float)qv, out_dt);
  const float d = qmm_round_dt(a - (float)z, out_dt);
  return d * sc;
}

// Dequantize; vector forms: runs of 4 (f32 out) or 8 (2-byte out), i.e. 16-byte stores, q aligned to a run, out to 16
// bytes, 1-byte q, total / 4 < 2^32.
// NT: streaming stores of out.  (A template: a branch around two forms of a store leaves the ordinary one.)
template <int OT, Form F, bool NT, bool FEW>
__global__ void __launch_bounds__(kThreads)
qdq_dequantize_kernel(const void* __restrict__ q, void* __restrict__ out, QdqParams p, QdqShape sh, int q_dt,
                      int int_subtract) {
  if constexpr (F != kAny) {
    constexpr int RUN = OT == XLA_AMD_DT_F32 ? 4 : 8, U = runs_per_thread<F, RUN, FEW>();
    const Runs<F, RUN, U> at(sh);
    if (!at.any) return;
    const RunParams<F, RUN, U> par(p, sh, at);
    uint32_t raw[U][RUN / 4];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t run = at.run(u);
      if constexpr (RUN == 4) {
        raw[u][0] = ((const uint32_t*)q)[run];
      } else {
        const i32x2 v = ((const i32x2*)q)[run];
        raw[u][0] = (uint32_t)v[0]; raw[u][1] = (uint32_t)v[1];
      }
    }
    float scv[RUN];
    int zv[RUN];
    if constexpr (F == kAlong) {
#pragma unroll
      for (int i = 0; i < RUN; ++i) { scv[i] = par.along.scale_of(p, i); zv[i] = par.along.zp_of(p, i); }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t run = at.run(u);
      float sc = 0.f;
      int z = 0;
      if constexpr (F != kAlong) { sc = qdq_scale(p, par.of[u]); z = par.of[u].zp; }
      float r[RUN];
#pragma unroll
      for (int i = 0; i < RUN; ++i) {
        const uint32_t b = (raw[u][i / 4] >> (8 * (i % 4))) & 0xffu;
        const int qv = q_dt == XLA_AMD_QDT_I8 ? (int)(int8_t)b : (int)b;
        if constexpr (F == kAlong) { sc = scv[i]; z = zv[i]; }
        r[i] = dequantize_value(qv, z, sc, OT, int_subtract);
      }
      if constexpr (OT == XLA_AMD_DT_F32) {
        const f32x4 v = {r[0], r[1], r[2], r[3]};
        if constexpr (NT) __builtin_nontemporal_store(v, (f32x4*)out + run);
        else ((f32x4*)out)[run] = v;
      } else {
        i32x4 pk;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          pk[i] = (int)(OT == XLA_AMD_DT_BF16 ? qmm_f32x2_to_bf16x2(r[2 * i], r[2 * i + 1]) : qmm_f32x2_to_f16x2(r[2 * i], r[2 * i + 1]));
        if constexpr (NT) __builtin_nontemporal_store(pk, (i32x4*)out + run);
        else ((i32x4*)out)[run] = pk;
      }
    }
  } else {
    const int64_t t = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (t >= sh.total) return;
    const uint32_t c = element_channel(sh, t);
    qmm_store(out, t, dequantize_value(qdq_load_q(q, t, q_dt), element_zp(p, c), qdq_factor(p, qmm_load(p.scale, c, p.scale_dt)), OT, int_subtract), OT);
  }
}

int qdt_size(int q_dt) { return q_dt == XLA_AMD_QDT_I16 ? 2 : q_dt == XLA_AMD_QDT_I32 ? 4 : 1; }
bool valid_qdt(int q_dt) { return q_dt >= XLA_AMD_QDT_I8 && q_dt <= XLA_AMD_QDT_I32; }

// Tensors that pass through the 256 MB Infinity Cache without staying in it are streamed past it, so that the other
// side of the call keeps its place: a float input larger than the cache (14336 x 14336 f32, 822 MB, and its f32 result:
// 355 us a pair with its loads kept, 314 streamed; 117 MB of bf16: 77 kept, 80 streamed), a float result of a quarter of
// it and more (235 MB of f32: 89 kept, 77 streamed; 117 MB of bf16: 63, 60).
constexpr int64_t kStreamIn = 256ll << 20, kStreamOut = 64ll << 20;

// The form for runs of `run` elements, and whether everything is aligned for it.
Form choose_form(const QdqShape& sh, int run, bool aligned) {
  if (!aligned || sh.total % run != 0 || sh.total / run > 0xffffffffLL - kPerBlock || sh.channels > 0x7fffffffLL) return kAny;
  if (sh.channels == 1) return kOne;
  if (sh.inner % run == 0 && sh.inner / run <= 0x7fffffffLL) return kRow;
  // (one row has nothing to share, and below 256 K elements a thread's eight channels take longer than eight threads:
  // a bf16 pair over 1 x 16.8 M 77 us element by element, 94 so, over 8 x 14336 4.8, 5.8)
  if (sh.inner == 1 && sh.channels % run == 0 && sh.outer > 1 && sh.outer <= 0x7fffffffLL && sh.total >= (1 << 18)) return kAlong;
  return kAny;
}

// Calls go(form constant, whether one run per thread, grid) for runs of `run` elements; returns the launch's status.
template <class Go>
int launch_form(Form f, const QdqShape& sh, int run, const char* what, Go&& go) {
  auto blocks_of = [&](int64_t u) -> int64_t {  // ... with u runs per thread
    if (f == kAny) return (sh.total + kThreads - 1) / kThreads;
    if (f == kAlong) return ((sh.outer + u - 1) / u * (sh.channels / run) + kThreads - 1) / kThreads;
    return (sh.total / run + kThreads * u - 1) / (kThreads * u);
  };
  const int64_t many = f == kAlong ? kDown : kPerBlock / (kThreads * run);
  const bool few = blocks_of(many) < (f == kAlong ? kFillAlong : kFill);
  const int64_t blocks = blocks_of(few ? 1 : many);
  if (blocks > 0x7fffffffLL) return qmm_fail(XLA_AMD_QMM_EUNSUPPORTED, "%s: tensor too large", what);
  const dim3 grid((unsigned)blocks);
  switch (f) {
    case kOne: go(qmm_const<kOne>{}, few, grid); break;
    case kRow: go(qmm_const<kRow>{}, few, grid); break;
    case kAlong: go(qmm_const<kAlong>{}, few, grid); break;
    default: go(qmm_const<kAny>{}, few, grid); break;
  }
  return QMM_CHECK_LAUNCH(what);
}

// Tensors of more elements than this go in pieces, which keeps runs and grids within 32 bits (and far from their cost).
constexpr int64_t kPiece = 1ll << 33;

// Calls piece(outer, channels, inner, parameters, first element) for a tensor of more than kPiece elements, cut along its
// first dimension of more than one entry; a piece may still be too large, along the next one.
template <class Piece>
int in_pieces(const QdqParams& p, int64_t outer, int64_t channels, int64_t inner, Piece&& piece) {
  if (channels == 1) { inner *= outer; outer = 1; }
  int64_t& cut = outer > 1 ? outer : channels > 1 ? channels : inner;
  const int64_t all = cut, rest = outer * channels * inner / all, most = kPiece / rest > 0 ? kPiece / rest : 1;
  const bool along = &cut == &channels;
  for (int64_t at = 0; at < all; at += most) {
    cut = all - at < most ? all - at : most;
    QdqParams pp = p;
    if (along) {
      pp.scale = (const char*)p.scale + at * qmm_dt_size(p.scale_dt);
      if (p.zp) pp.zp = (const char*)p.zp + at * (p.zp64 ? 8 : 4);
    }
    const int rc = piece(outer, channels, inner, pp, at * rest);
    if (rc != XLA_AMD_QMM_OK) return rc;
  }
  return XLA_AMD_QMM_OK;
}

int quantize(const char* what, const void* x, void* q, const QdqParams& p, int64_t outer, int64_t channels,
             int64_t inner, int x_dt, int q_dt, int32_t qmin, int32_t qmax, void* stream) {
  if (!x || !q || !p.scale || !p.zp) return qmm_fail(XLA_AMD_QMM_EINVAL, "%s: null pointer", what);
  if (outer < 0 || channels <= 0 || inner < 0) return qmm_fail(XLA_AMD_QMM_EINVAL, "%s: bad sizes", what);
  if (!qmm_valid_dt(x_dt) || !qmm_valid_dt(p.scale_dt) || !valid_qdt(q_dt) || qmin > qmax)
    return qmm_fail(XLA_AMD_QMM_EINVAL, "%s: bad dtype enum or bounds", what);
  const QdqShape sh = {outer * channels * inner, outer, channels, inner};
  if (sh.total == 0) return XLA_AMD_QMM_OK;
  if (sh.total > kPiece)
    return in_pieces(p, outer, channels, inner, [&](int64_t o, int64_t c, int64_t i, const QdqParams& pp, int64_t first) {
      return quantize(what, (const char*)x + first * qmm_dt_size(x_dt), (char*)q + first * qdt_size(q_dt), pp, o, c, i, x_dt, q_dt, qmin, qmax, stream);
    });
  const bool aligned = (q_dt == XLA_AMD_QDT_I8 || q_dt == XLA_AMD_QDT_U8) && (((uintptr_t)x & 15) == 0) && (((uintptr_t)q & 7) == 0);
  const bool nt = sh.total * qmm_dt_size(x_dt) > kStreamIn;
  return launch_form(choose_form(sh, 8, aligned), sh, 8, what, [&](auto fc, bool few, dim3 grid) {
    constexpr Form F = (Form)(int)fc;
    constexpr bool V = F != kAny;  // (element by element there is one kernel)
    const auto go = [&](auto kern) {
      hipLaunchKernelGGL(kern, grid, dim3(kThreads), 0, (hipStream_t)stream, x, q, p, sh, q_dt, (float)qmin, (float)qmax);
    };
    // (a tensor large enough to be streamed has many runs)
    const auto pick = [&](auto dc) {
      if (V && few) go(qdq_quantize_kernel<(int)dc, F, false, V>);
      else if (nt) go(qdq_quantize_kernel<(int)dc, F, V, false>);
      else go(qdq_quantize_kernel<(int)dc, F, false, false>);
    };
    if (x_dt == XLA_AMD_DT_BF16) pick(qmm_const<XLA_AMD_DT_BF16>{});
    else if (x_dt == XLA_AMD_DT_F16) pick(qmm_const<XLA_AMD_DT_F16>{});
    else pick(qmm_const<XLA_AMD_DT_F32>{});
  });
}

int dequantize(const char* what, const void* q, void* out, const QdqParams& p, int64_t outer, int64_t channels,
               int64_t inner, int q_dt, int out_dt, int int_subtract, void* stream) {
  if (!q || !out || !p.scale) return qmm_fail(XLA_AMD_QMM_EINVAL, "%s: null pointer", what);
  if (outer < 0 || channels <= 0 || inner < 0) return qmm_fail(XLA_AMD_QMM_EINVAL, "%s: bad sizes", what);
  if (!qmm_valid_dt(out_dt) || !qmm_valid_dt(p.scale_dt) || !valid_qdt(q_dt))
    return qmm_fail(XLA_AMD_QMM_EINVAL, "%s: bad dtype enum", what);
  const QdqShape sh = {outer * channels * inner, outer, channels, inner};
  if (sh.total == 0) return XLA_AMD_QMM_OK;
  if (sh.total > kPiece)
    return in_pieces(p, outer, channels, inner, [&](int64_t o, int64_t c, int64_t i, const QdqParams& pp, int64_t first) {
      return dequantize(what, (const char*)q + first * qdt_size(q_dt), (char*)out + first * qmm_dt_size(out_dt), pp, o, c, i, q_dt, out_dt, int_subtract, stream);
    });
  const int run = out_dt == XLA_AMD_DT_F32 ? 4 : 8;
  const bool aligned = (q_dt == XLA_AMD_QDT_I8 || q_dt == XLA_AMD_QDT_U8) && (((uintptr_t)q & (run - 1)) == 0) && (((uintptr_t)out & 15) == 0);
  const bool nt = sh.total * qmm_dt_size(out_dt) > kStreamOut;
  return launch_form(choose_form(sh, run, aligned), sh, run, what, [&](auto fc, bool few, dim3 grid) {
    constexpr Form F = (Form)(int)fc;
    constexpr bool V = F != kAny;  // (element by element there is one kernel)
    const auto go = [&](auto kern) {
      hipLaunchKernelGGL(kern, grid, dim3(kThreads), 0, (hipStream_t)stream, q, out, p, sh, q_dt, int_subtract);
    };
    const auto pick = [&](auto dc) {
      if (V && few) go(qdq_dequantize_kernel<(int)dc, F, false, V>);
      else if (nt) go(qdq_dequantize_kernel<(int)dc, F, V, false>);
      else go(qdq_dequantize_kernel<(int)dc, F, false, false>);
    };
    if (out_dt == XLA_AMD_DT_BF16) pick(qmm_const<XLA_AMD_DT_BF16>{});
    else if (out_dt == XLA_AMD_DT_F16) pick(qmm_const<XLA_AMD_DT_F16>{});
    else pick(qmm_const<XLA_AMD_DT_F32>{});
  });
}

}  // namespace

extern "C" int xla_amd_qmm_quantize_affine(const void* x, void* q, const float* inv_scale, const int32_t* zp,
                                           int64_t outer, int64_t channels, int64_t inner, int x_dt, int q_dt,
                                           int32_t qmin, int32_t qmax, void* stream) {
  return quantize("quantize_affine", x, q, QdqParams{inv_scale, zp, XLA_AMD_DT_F32, 0, 0}, outer, channels, inner, x_dt,
                  q_dt, qmin, qmax, stream);
}

extern "C" int xla_amd_qmm_dequantize_affine(const void* q, void* out, const float* scale, const int32_t* zp,
                                             int64_t outer, int64_t channels, int64_t inner, int q_dt, int out_dt,
                                             int int_subtract, void* stream) {
  return dequantize("dequantize_affine", q, out, QdqParams{scale, zp, XLA_AMD_DT_F32, 0, 0}, outer, channels, inner,
                    q_dt, out_dt, int_subtract, stream);
}

extern "C" int xla_amd_qmm_quantize_channels(const void* x, void* q, const void* scale, const void* zp, int64_t outer,
                                             int64_t channels, int64_t inner, int x_dt, int q_dt, int scale_dt,
                                             int zp_int64, int32_t qmin, int32_t qmax, void* stream) {
  return quantize("quantize_channels", x, q, QdqParams{scale, zp, scale_dt, zp_int64 != 0, 1}, outer, channels, inner,
                  x_dt, q_dt, qmin, qmax, stream);
}

extern "C" int xla_amd_qmm_dequantize_channels(const void* q, void* out, const void* scale, const void* zp,
                                               int64_t outer, int64_t channels, int64_t inner, int q_dt, int out_dt,
                                               int scale_dt, int zp_int64, void* stream) {
  return dequantize("dequantize_channels", q, out, QdqParams{scale, zp, scale_dt, zp_int64 != 0, 0}, outer, channels,
                    inner, q_dt, out_dt, 1, stream);
}
