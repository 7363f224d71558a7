// Building blocks of the paged attention kernels that keep full fp32 precision for any storage
// type on the matrix cores of gfx950, with no LDS between memory and the MFMA operands.
//
// The pool's rows are [d][token], so a 16-byte vector of a row is TV = 4 (fp32) or 8 (16-bit)
// consecutive tokens of one d. A tile is 16 vectors (64 or 128 tokens), vector x = tokens
// TV x .. TV x + TV - 1. With lane l, kd = l / 16, n16 = l % 16:
//   K: lane l loads vector 4 (n16 % 4) + n16 / 4 of rows d = 4 i + kd.
//   V: lane l loads vectors 4 u + kd of rows d = 16 nb + n16.
// Either load covers whole 128-byte lines: 4 consecutive K rows of each page (16-token pages:
// 256 bytes per page in fp32, 128 in 16 bits), or 16 V rows of one page (two in 16 bits). That is
// the decode kernel's order, whose tiles come from HBM, once. The multi-row kernel, whose tiles
// come from L2, takes K vector n16 and V vectors 4 kd + u instead (4 v + kd and 4 u + kd below
// become 4 kd + v and 4 kd + u): its K loads then cost 0.8 times as much, neighbouring lanes
// reading neighbouring vectors, while its V loads are spread over four pages each, which costs
// nothing there. In the decode kernel that order measured 60.8 -> 106.7 us (32 sequences, fp32).
//
// fp32 storage, v_mfma_f32_16x16x4_f32 (A: lane l holds A[n16][kd]; B: B[kd][n16]; C: lane l
// holds C[4 kd + v][n16]):
//   S^T = K . Q^T  component c of K row i is the A operand of product (i, c), whose row n16 is
//                  token TV x + c; B is q[row n16][4 i + kd]. Lane l then holds in s[c][v] the
//                  score of q row n16 for token TV (4 v + kd) + c (output row 4 kd + v is lane
//                  row n16 = 4 kd + v, whose vector is 4 v + kd).
//   O += P . V     component c of V vector (u, nb) is the B operand of product (u, c, nb), whose
//                  k slot kd is token TV (4 u + kd) + c: the token of s[c][u], so A is that
//                  register as it stands.
// 16-bit storage, v_mfma_f32_16x16x32 (A: lane l holds A[n16][8 kd .. + 7]; B: B[8 kd .. + 7][n16];
// C as above), whose products of 16-bit values are exact in fp32:
//   S^T = K . Q^T  k slot 8 kd + e of product (I, c) is row d = 4 (8 I + e) + kd, so A is
//                  component c of the lane's K rows 8 I .. 8 I + 7 (four v_perm_b32) and B the
//                  same elements of q row n16. The scores come out in the same places.
//   O += P . V     a V vector is a whole B operand (k slot 8 kd + e is token 8 (4 u + kd) + e) and
//                  A the eight probabilities s[0..7][u], as the sum of three 16-bit terms that
//                  carry all 24 bits of an fp32 value (split3): three products instead of the
//                  eight 16x16x4 ones that widened V would take, each of them half as long.
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
};

__device__ __forceinline__ f32x4_t mfma_f32(float a, float b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// component c (compile-time after unrolling) of an fp32 vector
__device__ __forceinline__ float comp(const uint4& x, int c) {
  return __uint_as_float(c == 0 ? x.x : c == 1 ? x.y : c == 2 ? x.z : x.w);
}
__device__ __forceinline__ uint32_t word(const uint4& x, int w) {
  return w == 0 ? x.x : w == 1 ? x.y : w == 2 ? x.z : x.w;
}

// s += K . Q^T over the 16 K rows of kr (fp32: summed in fours of them, so that a score is not one
// chain of D additions); q: the lane's q elements of those rows in LDS (fp32: 16
// floats; 16-bit: 16 raw elements), 16-byte aligned
template <int DT>
__device__ __forceinline__ void qk(const uint4 (&kr)[16], const void* q,
                                   f32x4_t (&s)[Vec<DT>::TV]) {
  const uint4* qv = reinterpret_cast<const uint4*>(q);
  if constexpr (DT == PIA_DTYPE_F32) {
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
      const uint4 x = qv[i4];
#pragma unroll
      for (int c0 = 0; c0 < 4; c0 += 2) {
        __builtin_amdgcn_sched_barrier(0);  // one pair of sums at a time (registers)
        f32x4_t t[2] = {f32x4_t{0.f, 0.f, 0.f, 0.f}, f32x4_t{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int c = 0; c < 2; ++c)
            t[c] = mfma_f32(comp(kr[4 * i4 + j], c0 + c), comp(x, j), t[c]);
#pragma unroll
        for (int c = 0; c < 2; ++c) s[c0 + c] += t[c];
      }
    }
  } else {
#pragma unroll
    for (int I = 0; I < 2; ++I) {
      __builtin_amdgcn_sched_barrier(0);  // one q chunk and its operands at a time (registers)
      const uint4 x = qv[I];
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        uint32_t a[4];
#pragma unroll
        for (int f = 0; f < 4; ++f) {
          const uint32_t r0 = word(kr[8 * I + 2 * f], c >> 1);
          const uint32_t r1 = word(kr[8 * I + 2 * f + 1], c >> 1);
          a[f] = __builtin_amdgcn_perm(r1, r0, (c & 1) ? 0x07060302u : 0x05040100u);
        }
        s[c] = tile::mfma16<DT>(make_uint4(a[0], a[1], a[2], a[3]), x, s[c]);
      }
    }
  }
}

// Eight fp32 probabilities s[0..7][u] as the sum of three 16-bit operands, each term what the ones
// before leave, rounded toward zero. A positive value has three positive terms (a zero one becomes
// the smallest denormal): times an infinite V they then give that infinity, as the value itself
// would, and not infinity - infinity or 0 times infinity. Three bf16 terms hold the 24 bits of an
// fp32 value, and the smallest denormal is 2^-133. Three fp16 terms hold them for values of
// 2^-1 .. 2^15; the caller scales the probabilities by kSplitShift, so the terms of a value are
// together between 2^-39 too small (what is below the last denormal) and 3 * 2^-39 too large (three
// filled terms) of the largest probability, and the row sum is that of the values themselves. So a
// row's outputs are too large by at most its number of keys times 3 * 2^-39 of the largest |V|: 4.5e-8
// at 8192 keys, all of them far below the largest.
template <int DT>
constexpr float kSplitShift = DT == PIA_DTYPE_F16 ? 15.f : 0.f;  // log2 units
template <int DT>
__device__ __forceinline__ void split3(const f32x4_t (&s)[8], int u, uint4 (&t)[3]) {
  uint32_t w[3][4];
#pragma unroll
  for (int f = 0; f < 4; ++f) {
    float a = s[2 * f][u], b = s[2 * f + 1][u];
    const uint32_t low =
        min(__float_as_uint(a), 1u) | (min(__float_as_uint(b), 1u) << 16);  // 1 where positive
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      if constexpr (DT == PIA_DTYPE_F16) {
        const auto h = __builtin_amdgcn_cvt_pkrtz(a, b);
        w[k][f] = __builtin_bit_cast(uint32_t, h);
        a -= float(h[0]);
        b -= float(h[1]);
      } else {
        w[k][f] = __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
        a -= bf16_hi(__float_as_uint(a));
        b -= bf16_hi(__float_as_uint(b));
      }
      if (k > 0 || DT == PIA_DTYPE_F16) {  // a zero term of a positive value: the smallest one
        typedef unsigned short u16x2_t __attribute__((ext_vector_type(2)));
        w[k][f] = __builtin_bit_cast(
            uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2_t, w[k][f]),
                                                __builtin_bit_cast(u16x2_t, low)));
      }
    }
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) t[k] = make_uint4(w[k][0], w[k][1], w[k][2], w[k][3]);
}

// O += P . V over the V vectors u0 .. u0 + NU - 1 (vr[nb * NU + u - u0]), NB blocks of 16 d. fp32:
// the vectors' products are summed on their own first, two blocks at a time, so that a long
// context is not one chain of additions.
template <int DT, int NB, int NU>
__device__ __forceinline__ void pv(const uint4 (&vr)[NB * NU], const f32x4_t (&p)[Vec<DT>::TV],
                                   int u0, f32x4_t (&acc)[NB]) {
  if constexpr (DT == PIA_DTYPE_F32) {
#pragma unroll
    for (int n0 = 0; n0 < NB; n0 += 2) {
      __builtin_amdgcn_sched_barrier(0);  // one pair at a time (registers)
      f32x4_t t[2] = {f32x4_t{0.f, 0.f, 0.f, 0.f}, f32x4_t{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int u = 0; u < NU; ++u)
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
          for (int j = 0; j < 2; ++j)
            t[j] = mfma_f32(p[c][u0 + u], comp(vr[(n0 + j) * NU + u], c), t[j]);
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        acc[n0 + j] += t[j];
        asm volatile("" : "+v"(acc[n0 + j]));  // added now: delayed, the sums were spilled
      }
    }
  } else {
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      __builtin_amdgcn_sched_barrier(0);  // one set of terms at a time (registers)
      uint4 t[3];
      split3<DT>(p, u0 + u, t);
#pragma unroll
      for (int k = 0; k < 3; ++k)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) acc[nb] = tile::mfma16<DT>(t[k], vr[nb * NU + u], acc[nb]);
    }
  }
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
