// RMSNorm (with the residual add before it) and the per-head RMSNorm + RoPE of a decode step.
//
// The reference's formulas (src/plastic_infer/exec/attention.py:53-95: x / sqrt(mean(x^2) + eps)
// times the weight; rotate-half RoPE from table rows), each as one pass with fp32 arithmetic and
// one rounding of the result (the sum of the add is rounded first, as a tensor of its own would
// be). At decode sizes these calls are all launch latency: as separate elementwise operations
// one norm is six launches, and norm + RoPE of q and k some twenty. A step of two layers, 64
// sequences, hidden 2048: 1441 -> 1024 us with one launch each (3.0-4.6 us).
#include "pia_internal.h"

namespace pia {
namespace {

constexpr int RN_THREADS = 256;

// Sum of v over the workgroup (every thread receives it).
__device__ __forceinline__ float block_sum(float v) {
  __shared__ float part[RN_THREADS / 64];
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
  __syncthreads();
  float s = 0.f;
#pragma unroll
  for (int w = 0; w < RN_THREADS / 64; ++w) s += part[w];
  return s;
}

// One workgroup per row of n elements: s = x (+ y, rounded and written to sum), then
// out = s / sqrt(mean(s^2) + eps) * w. A thread reads back only what it wrote itself.
template <int DT, bool ADD, bool VEC>
__global__ __launch_bounds__(RN_THREADS) void rms_norm_kernel(
    typename Elem<DT>::T* __restrict__ out, typename Elem<DT>::T* sum,
    const typename Elem<DT>::T* x, const typename Elem<DT>::T* __restrict__ y,
    const typename Elem<DT>::T* __restrict__ w, int n, float eps) {
  using El = Elem<DT>;
  using T = typename El::T;
  constexpr int V = VEC ? 16 / int(sizeof(T)) : 1;
  struct alignas(V * sizeof(T)) Pack {
    T v[V];
  };
  const int64_t r = int64_t(blockIdx.x) * n;
  float sq = 0.f;
  for (int i = threadIdx.x * V; i < n; i += RN_THREADS * V) {
    Pack a = *reinterpret_cast<const Pack*>(x + r + i);
    if constexpr (ADD) {
      const Pack b = *reinterpret_cast<const Pack*>(y + r + i);
#pragma unroll
      for (int j = 0; j < V; ++j) El::store(a.v, j, El::load(a.v, j) + El::load(b.v, j));
      *reinterpret_cast<Pack*>(sum + r + i) = a;
    }
#pragma unroll
    for (int j = 0; j < V; ++j) sq += El::load(a.v, j) * El::load(a.v, j);
  }
  const float root = sqrtf(block_sum(sq) / float(n) + eps);
  const T* s = ADD ? sum : x;
  for (int i = threadIdx.x * V; i < n; i += RN_THREADS * V) {
    const Pack a = *reinterpret_cast<const Pack*>(s + r + i);
    const Pack g = *reinterpret_cast<const Pack*>(w + i);
    Pack o;
#pragma unroll
    for (int j = 0; j < V; ++j) El::store(o.v, j, El::load(a.v, j) / root * El::load(g.v, j));
    *reinterpret_cast<Pack*>(out + r + i) = o;
  }
}

// One wave per head of a row: q heads first, then k heads. Element d < D / 2 and its partner
// d + D / 2 sit in one lane. cos / sin: the rows' own table rows [rows, D].
template <int DT, bool NORM>
__global__ __launch_bounds__(256) void qk_norm_rope_kernel(
    typename Elem<DT>::T* __restrict__ q_out, typename Elem<DT>::T* __restrict__ k_out,
    const typename Elem<DT>::T* __restrict__ q, const typename Elem<DT>::T* __restrict__ k,
    const typename Elem<DT>::T* __restrict__ qw, const typename Elem<DT>::T* __restrict__ kw,
    const typename Elem<DT>::T* __restrict__ cos, const typename Elem<DT>::T* __restrict__ sin,
    int64_t rows, int Hq, int Hkv, int D, float eps) {
  using El = Elem<DT>;
  using T = typename El::T;
  const int lane = threadIdx.x & 63;
  const int64_t i = int64_t(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (i >= rows * (Hq + Hkv)) return;
  const int64_t b = i / (Hq + Hkv);
  const int h = int(i - b * (Hq + Hkv));
  const bool is_q = h < Hq;
  const int64_t at = is_q ? (b * Hq + h) * D : (b * Hkv + h - Hq) * D;
  const T* x = (is_q ? q : k) + at;
  T* o = (is_q ? q_out : k_out) + at;
  const T* w = is_q ? qw : kw;
  const int half = D / 2;
  float root = 1.f;
  if constexpr (NORM) {
    float sq = 0.f;
    for (int d = lane; d < D; d += 64) sq += El::load(x, d) * El::load(x, d);
    root = sqrtf(wave_sum(sq) / float(D) + eps);
  }
  for (int d = lane; d < half; d += 64) {
    float a = El::load(x, d), c = El::load(x, d + half);
    if constexpr (NORM) {
      a = a / root * El::load(w, d);
      c = c / root * El::load(w, d + half);
    }
    El::store(o, d, a * El::load(cos, b * D + d) - c * El::load(sin, b * D + d));
    El::store(o, d + half,
              c * El::load(cos, b * D + d + half) + a * El::load(sin, b * D + d + half));
  }
}

}  // namespace
}  // namespace pia

using namespace pia;

#define PIA_BY_DTYPE(dtype, CALL)                    \
  switch (dtype) {                                   \
    case PIA_DTYPE_F32: CALL(PIA_DTYPE_F32); break;  \
    case PIA_DTYPE_F16: CALL(PIA_DTYPE_F16); break;  \
    default: CALL(PIA_DTYPE_BF16); break;            \
  }

extern "C" int pia_rms_norm(void* out, void* sum, const void* x, const void* residual,
                            const void* weight, int64_t rows, int n, float eps, int dtype,
                            void* stream) {
  if (dtype != PIA_DTYPE_F32 && dtype != PIA_DTYPE_F16 && dtype != PIA_DTYPE_BF16)
    return fail(PIA_EUNSUPPORTED, "rms_norm: dtype must be bf16, fp16 or fp32");
  if (rows < 0 || n <= 0) return fail(PIA_EINVAL, "rms_norm: invalid size");
  if (rows == 0) return 0;
  if (rows > 0x7fffffff) return fail(PIA_EINVAL, "rms_norm: too many rows");
  if (!out || !x || !weight || (residual && !sum)) return fail(PIA_EINVAL, "rms_norm: null pointer");
  hipStream_t s = as_stream(stream);
  const int vec = dtype == PIA_DTYPE_F32 ? 4 : 8;
  const bool v16 = n % vec == 0 && aligned(out, 16) && aligned(x, 16) && aligned(weight, 16) &&
                   (!residual || (aligned(residual, 16) && aligned(sum, 16)));
#define PIA_RN3(DT, ADD, VEC)                                                              \
  hipLaunchKernelGGL((rms_norm_kernel<DT, ADD, VEC>), dim3(unsigned(rows)), dim3(RN_THREADS), 0, \
                     s, static_cast<Elem<DT>::T*>(out), static_cast<Elem<DT>::T*>(sum),    \
                     static_cast<const Elem<DT>::T*>(x),                                   \
                     static_cast<const Elem<DT>::T*>(residual),                            \
                     static_cast<const Elem<DT>::T*>(weight), n, eps)
#define PIA_RN(DT)                                              \
  if (residual) {                                               \
    if (v16) PIA_RN3(DT, true, true); else PIA_RN3(DT, true, false);   \
  } else {                                                      \
    if (v16) PIA_RN3(DT, false, true); else PIA_RN3(DT, false, false); \
  }
  PIA_BY_DTYPE(dtype, PIA_RN)
#undef PIA_RN
#undef PIA_RN3
  return check_launch("rms_norm");
}

extern "C" int pia_qk_norm_rope(void* q_out, void* k_out, const void* q, const void* k,
                                const void* q_weight, const void* k_weight, const void* cos,
                                const void* sin, int64_t rows, int num_heads, int num_kv_heads,
                                int head_dim, float eps, int dtype, void* stream) {
  if (dtype != PIA_DTYPE_F32 && dtype != PIA_DTYPE_F16 && dtype != PIA_DTYPE_BF16)
    return fail(PIA_EUNSUPPORTED, "qk_norm_rope: dtype must be bf16, fp16 or fp32");
  if (rows < 0 || num_heads < 0 || num_kv_heads < 0 || head_dim <= 0 || head_dim % 2)
    return fail(PIA_EINVAL, "qk_norm_rope: invalid size");
  const int64_t waves = rows * (int64_t(num_heads) + num_kv_heads);
  if (waves == 0) return 0;
  if (ceil_div(waves, 4) > 0x7fffffff) return fail(PIA_EINVAL, "qk_norm_rope: too many rows");
  if ((num_heads && (!q_out || !q)) || (num_kv_heads && (!k_out || !k)) || !cos || !sin ||
      !q_weight != !k_weight)
    return fail(PIA_EINVAL, "qk_norm_rope: null pointer");
  hipStream_t s = as_stream(stream);
#define PIA_QR2(DT, NORM)                                                                    \
  hipLaunchKernelGGL((qk_norm_rope_kernel<DT, NORM>), dim3(unsigned(ceil_div(waves, 4))),    \
                     dim3(256), 0, s, static_cast<Elem<DT>::T*>(q_out),                      \
                     static_cast<Elem<DT>::T*>(k_out), static_cast<const Elem<DT>::T*>(q),   \
                     static_cast<const Elem<DT>::T*>(k),                                     \
                     static_cast<const Elem<DT>::T*>(q_weight),                              \
                     static_cast<const Elem<DT>::T*>(k_weight),                              \
                     static_cast<const Elem<DT>::T*>(cos),                                   \
                     static_cast<const Elem<DT>::T*>(sin), rows, num_heads, num_kv_heads,    \
                     head_dim, eps)
#define PIA_QR(DT) \
  if (q_weight) PIA_QR2(DT, true); else PIA_QR2(DT, false)
  PIA_BY_DTYPE(dtype, PIA_QR)
#undef PIA_QR
#undef PIA_QR2
  return check_launch("qk_norm_rope");
}
