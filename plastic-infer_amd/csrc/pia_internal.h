// Internal helpers shared by the HIP translation units of libplastic_infer_amd.so (gfx950 only).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdarg.h>
#include <stdio.h>

#include "plastic_infer_amd.h"

namespace pia {

// Thread-local last-error text behind pia_last_error().
void set_error(const char* fmt, ...) __attribute__((format(printf, 1, 2)));

inline int fail(int code, const char* what) {
  set_error("%s", what);
  return code;
}

// Checks a HIP launch / runtime call; records the text and returns the hipError_t as int.
inline int check_hip(hipError_t e, const char* where) {
  if (e == hipSuccess) return 0;
  set_error("%s: %s", where, hipGetErrorString(e));
  return (int)e;
}

// Compute units of the current device (cached per device; 256 if the query fails).
int device_cus();

inline int check_launch(const char* where) { return check_hip(hipGetLastError(), where); }

inline hipStream_t as_stream(void* s) { return reinterpret_cast<hipStream_t>(s); }

inline bool aligned(const void* p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) % a) == 0; }

inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Multi-row paged attention on the matrix cores (paged_prefill.hip): whether a call takes it,
// and its launch (arguments already checked by pia_paged_attention).
bool prefill_mfma_path(int dtype, int Hq, int Hkv, int D, int P, int num_seqs,
                       int64_t total_q_rows, const int32_t* cu_q, float scale);
int launch_prefill_mfma(int dtype, void* out, const void* q, const void* k_pages,
                        const void* v_pages,
                        const int32_t* bt, int64_t bt_stride, const int32_t* kv_lens,
                        const int32_t* cu_q, const int32_t* offsets, int num_seqs,
                        int64_t total_q_rows, int Hq, int Hkv, int64_t num_pages,
                        float scale_log2, hipStream_t s);

// Paged attention of any rows with fp32 precision on the matrix cores (paged_rows.hip): whether a
// call takes it, and its launch (arguments already checked by pia_paged_attention).
bool rows_path(int dtype, int Hq, int Hkv, int D, int P, int num_seqs, int64_t total_q_rows,
               const void* k_pages, const void* v_pages);
int launch_rows(int dtype, void* out, const void* q, const void* k_pages, const void* v_pages,
                const int32_t* bt, int64_t bt_stride, const int32_t* kv_lens,
                const int32_t* cu_q, const int32_t* offsets, int num_seqs, int64_t total_q_rows,
                int Hq, int Hkv, int D, int P, int64_t num_pages, float scale_log2,
                hipStream_t s);

// pia_moe_expert_gemm with the number of experts that a layer's ids come from, where w holds more
// slots than that (0: not said).
int expert_gemm(void* out, const void* a, const void* w, const float* topk_weights,
                const int32_t* sorted_token_ids, const int32_t* expert_ids,
                const int32_t* num_tokens_post_pad, int64_t max_num_tokens_padded, int block_m,
                int64_t numel, int a_div, int64_t lda, int num_experts, int layer_experts,
                int n_rows, int k_dim, int64_t ldo, int activation, int mul_routed_weight,
                int dtype, void* workspace, int64_t workspace_bytes, void* stream);

// ---------------------------------------------------------------------------------------------
// Device helpers
// ---------------------------------------------------------------------------------------------

// Work list of the multi-row attention kernels: workgroup `block` (on XCD block % 8) of a call with
// n items per kv head takes item `j` of kv head `h`; false: none. An XCD runs whole heads where
// 8 divides their number. Else it shares heads with others: item by item, so that every XCD gets
// the same part of every sequence and sequences of different lengths do not load the XCDs
// differently, as contiguous runs of a sequence-major list did (2 sequences, 16/8 heads, fp32: 1.2
// of 2 waves per SIMD in flight); or, where the caller says that its sequences are alike (`runs`), in
// contiguous runs of the heads' items, so that K / V of most (sequence, head) go through one XCD's
// L2 and not all that share the head (4 prompts of 1024 behind 1000, 32/4 heads: 128.2 us item by
// item, 115.2 in runs).
__device__ __forceinline__ bool xcd_item(uint32_t block, int n, int Hkv, int& h, int& j,
                                         bool runs = false) {
  // log2 of the head classes (heads h with one remainder) and of the XCDs that share one
  const int own = Hkv % 8 == 0 ? 3 : Hkv % 4 == 0 ? 2 : Hkv % 2 == 0 ? 1 : 0, share = 3 - own;
  const uint32_t x = block & 7, k = block >> 3;
  const uint32_t all = uint32_t(Hkv >> own) * uint32_t(n);
  uint32_t l = (k << share) + (x >> own);
  if (runs) {
    const uint32_t run = (all + (1u << share) - 1) >> share;
    if (k >= run) return false;
    l = (x >> own) * run + k;
  }
  if (l >= all) return false;
  const uint32_t i = l / uint32_t(n);
  h = int(x & ((1u << own) - 1)) + int(i << own);
  j = int(l - i * uint32_t(n));
  return true;
}

// bf16 <-> f32 by bit manipulation (bf16 is the upper half of an IEEE binary32).
__device__ __forceinline__ float bf16_lo(uint32_t x) { return __uint_as_float(x << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t x) { return __uint_as_float(x & 0xffff0000u); }
__device__ __forceinline__ float bf16_to_f32(uint16_t x) { return __uint_as_float(uint32_t(x) << 16); }

// Round-to-nearest-even f32 -> bf16 (NaN kept quiet), same rounding as torch's .to(bfloat16).
__device__ __forceinline__ uint16_t f32_to_bf16(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return uint16_t((u >> 16) | 0x40u);
  u += 0x7fffu + ((u >> 16) & 1u);
  return uint16_t(u >> 16);
}

__device__ __forceinline__ float half_to_f32(uint16_t x) {
  return float(__builtin_bit_cast(_Float16, x));
}
__device__ __forceinline__ uint16_t f32_to_half(float f) {
  return __builtin_bit_cast(uint16_t, _Float16(f));  // round to nearest even
}

// Element load/store as f32 for the three storage types (dtype codes of the public header).
template <int DT> struct Elem;
template <> struct Elem<PIA_DTYPE_F32> {
  using T = float;
  __device__ __forceinline__ static float load(const T* p, int64_t i) { return p[i]; }
  __device__ __forceinline__ static void store(T* p, int64_t i, float v) { p[i] = v; }
};
template <> struct Elem<PIA_DTYPE_BF16> {
  using T = uint16_t;
  __device__ __forceinline__ static float load(const T* p, int64_t i) { return bf16_to_f32(p[i]); }
  __device__ __forceinline__ static void store(T* p, int64_t i, float v) { p[i] = f32_to_bf16(v); }
};
template <> struct Elem<PIA_DTYPE_F16> {
  using T = uint16_t;
  __device__ __forceinline__ static float load(const T* p, int64_t i) { return half_to_f32(p[i]); }
  __device__ __forceinline__ static void store(T* p, int64_t i, float v) { p[i] = f32_to_half(v); }
};

// Wave64 reductions through ds_swizzle/bpermute-backed shuffles.
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}

}  // namespace pia
