// Building blocks of the paged attention kernels that run on the fp32 matrix cores
// (v_mfma_f32_16x16x4_f32, gfx950) for any storage type: 16-bit K / V elements are widened in
// registers, probabilities and sums stay fp32.
//
// Operand layouts of v_mfma_f32_16x16x4_f32 (lane l, kd = l / 16, n16 = l % 16):
//   A (16 x 4): lane l holds A[n16][kd]      B (4 x 16): lane l holds B[kd][n16]
//   C (16 x 16): lane l holds C[4 kd + v][n16], v < 4
//
// The pool's rows are [d][token], so a 16-byte vector of a row is TV = 4 (fp32) or 8 (16-bit)
// consecutive tokens of one d, and K and V go from memory straight into MFMA operands, with no
// LDS: a tile is 16 vectors (64 or 128 tokens), vector x = tokens TV x .. TV x + TV - 1.
//   S^T = K . Q^T  lane l loads vector x = 4 (n16 % 4) + n16 / 4 of rows d = 4 i + kd; component
//                  c of it is the A operand of product (i, c), whose row n16 is token TV x + c;
//                  B is q[row n16][4 i + kd]. Lane l then holds, in s[c][v], the score of q row
//                  n16 for token TV (4 v + kd) + c (output row 4 kd + v is lane row n16 = 4 kd +
//                  v, whose vector is 4 v + kd).
//   O += P . V     lane l loads vector 4 u + kd of rows d = 16 nb + n16; component c is the B
//                  operand of product (u, c, nb), whose k slot kd is token TV (4 u + kd) + c: the
//                  token of s[c][u], so A is that register as it stands.
// Either load covers whole 128-byte lines: 4 consecutive K rows of each page (16-token pages:
// 256 bytes per page in fp32, 128 in 16 bits), or 16 V rows of one page (two in 16 bits).
#pragma once

#include "attn_tiles.h"
#include "pia_internal.h"

namespace pia {
namespace tile32 {

using tile::f32x4_t;
typedef uint32_t u32x4_nt __attribute__((ext_vector_type(4)));

template <int DT>
struct Vec {
  using T = typename Elem<DT>::T;
  static constexpr int TV = 16 / int(sizeof(T));  // tokens of a 16-byte vector
  static constexpr int TOKENS = 16 * TV;          // tokens of a tile
  // component c (compile-time after unrolling) of a vector, widened
  __device__ __forceinline__ static float get(const uint4& x, int c) {
    const uint32_t w = TV == 4 ? (c == 0 ? x.x : c == 1 ? x.y : c == 2 ? x.z : x.w)
                               : (c < 2 ? x.x : c < 4 ? x.y : c < 6 ? x.z : x.w);
    if constexpr (DT == PIA_DTYPE_F32) return __uint_as_float(w);
    else if constexpr (DT == PIA_DTYPE_F16)
      return half_to_f32(uint16_t((c & 1) ? (w >> 16) : (w & 0xffffu)));
    else return (c & 1) ? bf16_hi(w) : bf16_lo(w);
  }
  // components at or past n (n <= 0: all of them) become zero
  __device__ __forceinline__ static void keep_below(uint4& x, int n) {
    if constexpr (TV == 4) {
      x.x = n > 0 ? x.x : 0u;
      x.y = n > 1 ? x.y : 0u;
      x.z = n > 2 ? x.z : 0u;
      x.w = n > 3 ? x.w : 0u;
    } else {
      x.x = tile::mask_pair(x.x, 0, n);
      x.y = tile::mask_pair(x.y, 2, n);
      x.z = tile::mask_pair(x.z, 4, n);
      x.w = tile::mask_pair(x.w, 6, n);
    }
  }
  // component c (wave-uniform) := raw element bits v, on the lanes where own
  __device__ __forceinline__ static void put(uint4& x, int c, uint32_t v, bool own) {
    if constexpr (TV == 4) {
      x.x = own && c == 0 ? v : x.x;
      x.y = own && c == 1 ? v : x.y;
      x.z = own && c == 2 ? v : x.z;
      x.w = own && c == 3 ? v : x.w;
    } else {
      const uint32_t sh = (c & 1) ? 16u : 0u, keep = ~(0xffffu << sh), nv = v << sh;
      const int wd = c >> 1;
      x.x = own && wd == 0 ? ((x.x & keep) | nv) : x.x;
      x.y = own && wd == 1 ? ((x.y & keep) | nv) : x.y;
      x.z = own && wd == 2 ? ((x.z & keep) | nv) : x.z;
      x.w = own && wd == 3 ? ((x.w & keep) | nv) : x.w;
    }
  }
  // an element's raw bits
  __device__ __forceinline__ static uint32_t raw(const T* p) {
    if constexpr (DT == PIA_DTYPE_F32) return __float_as_uint(*p);
    else return *p;
  }
  __device__ __forceinline__ static float widen(uint32_t bits) {
    if constexpr (DT == PIA_DTYPE_F32) return __uint_as_float(bits);
    else if constexpr (DT == PIA_DTYPE_F16) return half_to_f32(uint16_t(bits));
    else return bf16_lo(bits);
  }
};

__device__ __forceinline__ f32x4_t mfma_f32(float a, float b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// scores += K . Q^T over N K vectors (rows 4 (i0 + i) + kd), q[i0 + i] the matching q elements
template <int DT, int N, int QN>
__device__ __forceinline__ void qk(const uint4 (&kr)[N], const float (&q)[QN], int i0,
                                   f32x4_t (&s)[Vec<DT>::TV]) {
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int c = 0; c < Vec<DT>::TV; ++c)
      s[c] = mfma_f32(Vec<DT>::get(kr[i], c), q[i0 + i], s[c]);
}

// O += P . V over the V vectors u0 .. u0 + NU - 1 (vr[nb * NU + u - u0]), NB blocks of 16 d
template <int DT, int NB, int NU>
__device__ __forceinline__ void pv(const uint4 (&vr)[NB * NU], const f32x4_t (&p)[Vec<DT>::TV],
                                   int u0, f32x4_t (&acc)[NB]) {
#pragma unroll
  for (int u = 0; u < NU; ++u)
#pragma unroll
    for (int c = 0; c < Vec<DT>::TV; ++c)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
        acc[nb] = mfma_f32(p[c][u0 + u], Vec<DT>::get(vr[nb * NU + u], c), acc[nb]);
}

// 16-byte non-temporal load (K / V read once per launch) or an ordinary one (read again by
// other work items, through L2)
template <bool NT, typename T>
__device__ __forceinline__ uint4 load16(const T* p) {
  if constexpr (NT) {
    const u32x4_nt v = __builtin_nontemporal_load(reinterpret_cast<const u32x4_nt*>(p));
    return make_uint4(v.x, v.y, v.z, v.w);
  } else {
    return *reinterpret_cast<const uint4*>(p);
  }
}

// Sum over lanes l, l ^ 16, l ^ 32, l ^ 48 (the four lanes that hold one q row's scores).
__device__ __forceinline__ float sum_col4(float v) {
  const unsigned u = __float_as_uint(v);
  const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  const float m = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const unsigned w = __float_as_uint(m);
  const auto b = __builtin_amdgcn_permlane32_swap(w, w, false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

}  // namespace tile32
}  // namespace pia
