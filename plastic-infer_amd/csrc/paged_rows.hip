// Paged attention of any number of query rows per sequence with fp32 precision throughout, on the
// matrix cores of gfx950: any storage type (fp32, fp16, bf16), head_dim 64 or 128, any Hq / Hkv,
// page sizes that are whole 16-byte vectors, optional causal offsets. Takes the calls that
// paged_prefill_mfma does not.
//
// Work item (one workgroup of four waves): one kv head and 16 consecutive (position, q head) rows
// of one sequence: flat row R is position R / G, head h * G + R % G, so every group size fills the
// 16-row MFMA blocks. The item's keys are walked in tiles of 16 vectors (64 fp32 or 128 16-bit
// tokens); wave w takes tiles w, w + 4, ..., with its own running max, sum and accumulators, K and
// V coming from memory straight into MFMA operands a tile ahead (layouts and products in
// attn_tiles_f32.h). The four waves' partials are merged in LDS at the end. Splitting the keys
// over the waves, not the rows, keeps short prompts' few row blocks on four times the SIMDs and
// needs no barrier in the loop. fp32 pools are bound by the 16x16x4 products (32 cycles for 2048
// FLOP); 16-bit pools by the tile reads from L2: 64 KiB (D = 128) for each 16 rows and tile.
// Work list as in paged_prefill_mfma: the items of one (sequence, kv head) run on one XCD or few,
// whose L2 holds its K / V.
//
// A row sees keys below its own limit; the other keys of a tile score -inf. Tokens that no row of
// the item sees have their V components zeroed. A token that only some of the rows see may hold a
// non-finite V, which the others' zero probabilities would turn into NaN: such a tile part (on
// the causal boundary only) is summed on the vector ALU, row by row.
//
// Measured against paged_attention_tiled, which ran a workgroup per row: 2 sequences of 300..600
// rows behind 0..512 tokens, 16/8 heads of 128, fp32:
// 743 -> 116 us, 98 us with the heads dealt to the XCDs, 93 us with the K loads' lanes in the order
// of their vectors (8 sequences of 1024 rows behind 3072, 28/4 heads, bf16: 23.3 ms, 1964, then 1504
// us), 83 us with the sums in pairs (attn_tiles_f32.h). Two
// 16-row blocks per wave, which halve the tile reads: 88 and 1535 us, and 28.6 against 23.0 us for
// 2 short ones at head_dim 64; not kept.
#include <algorithm>

#include "attn_tiles.h"
#include "attn_tiles_f32.h"
#include "pia_internal.h"

namespace pia {
namespace {

using tile::f32x4_t;

constexpr int PR_WAVES = 4;
constexpr int PR_ROWS = 16;
constexpr int PR_MAX_SEQS = 1024;  // sequences per launch (item prefix in LDS)

__device__ __forceinline__ bool nonfinite16(uint32_t bits, int dt) {
  const uint32_t e = dt == PIA_DTYPE_F16 ? 0x7c00u : 0x7f80u;
  return (bits & e) == e;
}

template <int DT, int D>
__global__ __launch_bounds__(64 * PR_WAVES, 2) void paged_attention_rows(
    typename Elem<DT>::T* __restrict__ out, const typename Elem<DT>::T* __restrict__ q,
    const typename Elem<DT>::T* __restrict__ kpool, const typename Elem<DT>::T* __restrict__ vpool,
    const int32_t* __restrict__ bt, int64_t bt_stride, const int32_t* __restrict__ kv_lens,
    const int32_t* __restrict__ cu_q, const int32_t* __restrict__ offsets, int B,
    int total_rows, int Hkv, int G, int P, int64_t num_pages, float scale_log2) {
  using T = typename Elem<DT>::T;
  using V = tile32::Vec<DT>;
  constexpr int TV = V::TV, TOK = V::TOKENS, NB = D / 16, NI = D / 4;
  constexpr int NU = D == 128 ? 2 : 4;          // V vectors u of one register buffer
  constexpr int QS = NI + 16 / int(sizeof(T));  // LDS stride of a lane's q elements
  constexpr int NT = 64 * PR_WAVES;
  __shared__ int item_pref[PR_MAX_SEQS + 1];
  __shared__ int wsum[PR_WAVES];
  __shared__ __align__(16) T qs[64 * QS];  // [lane]: q[row n16][4 i + kd] (fp32: pre-scaled)
  // per wave: row by row sums' probabilities [16][TS], at the end the partials [16][DS]: D
  // unnormalised outputs, running max, sum
  constexpr int TS = 4 * NU * TV + 1, DS = D + 3;
  __shared__ float part[PR_WAVES][PR_ROWS * (TS > DS ? TS : DS)];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // see paged_decode_f32: lane terms recomputed at each use instead of kept and spilled
  auto lane_now = [&]() -> int {
    int l = lane;
    asm volatile("" : "+v"(l));
    return l;
  };
  const int Hq = Hkv * G;

  // rows of sequence b: cu_q[b] .. cu_q[b + 1], the last one's to the end of q
  auto rows_of = [&](int b) {
    if (!cu_q) return 1;
    return (b == B - 1 ? total_rows : min(cu_q[b + 1], total_rows)) - cu_q[b];
  };
  if (tid == 0) item_pref[0] = 0;
  int carry = 0;
  for (int c0 = 0; c0 < B; c0 += NT) {
    const int i = c0 + tid;
    const int n = i < B ? rows_of(i) : 0;
    int incl = n > 0 ? (n * G + PR_ROWS - 1) / PR_ROWS : 0;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(incl, o, 64);
      if (lane >= o) incl += y;
    }
    if (lane == 63) wsum[wave] = incl;
    __syncthreads();
    int base = carry;
    for (int x = 0; x < wave; ++x) base += wsum[x];
    if (i < B) item_pref[i + 1] = base + incl;
#pragma unroll
    for (int x = 0; x < PR_WAVES; ++x) carry += wsum[x];
    __syncthreads();
  }
  // this workgroup's item: its kv head, and item j of that head over the sequences in order
  int h, j;
  if (!xcd_item(blockIdx.x, carry, Hkv, h, j)) return;
  int lo = 0, hi = B - 1;  // the sequence holding the item: the last with item_pref[b] <= j
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (item_pref[mid] <= j) lo = mid; else hi = mid - 1;
  }
  const int b = lo;
  const int R0 = (item_pref[b + 1] - 1 - j) * PR_ROWS;  // the last rows, with the most keys, first
  const int64_t row0 = cu_q ? int64_t(cu_q[b]) : int64_t(b);
  const int n_rows = rows_of(b) * G;  // flat rows of the (sequence, kv head)
  int kv_len = kv_lens[b];
  kv_len = kv_len < 0 ? 0 : (int64_t(kv_len) > bt_stride * P ? int(bt_stride * P) : kv_len);
  const int off = offsets ? offsets[b] : 0;
  auto limit_of = [&](int R) -> int {  // keys that flat row R sees
    if (R >= n_rows) return 0;
    return offsets ? max(0, min(kv_len, off + R / G + 1)) : kv_len;
  };
  const int R_last = min(R0 + PR_ROWS, n_rows) - 1;
  const int kmax = limit_of(R_last), kmin = limit_of(R0);  // limits rise with the position
  const int lim = limit_of(R0 + (lane & 15));
  const int npages = (kv_len + P - 1) / P;
  const int ntiles = (kmax + TOK - 1) / TOK;
  const int32_t* btb = bt + int64_t(b) * bt_stride;

  // q rows of the item: element (r, d) to qs[(d % 4) * 16 + r][d / 4]
  for (int e = tid; e < PR_ROWS * D; e += NT) {
    const int r = e / D, d = e % D, R = R0 + r;
    T x = T(0);
    if (R < n_rows)
      x = q[(row0 + R / G) * Hq * D + int64_t(h * G + R % G) * D + d];
    if constexpr (DT == PIA_DTYPE_F32) x *= scale_log2;
    qs[((d & 3) * 16 + r) * QS + (d >> 2)] = x;
  }
  __syncthreads();

  const int vpp = P / TV;  // vectors per page row
  auto load_bt = [&](int t) -> int {  // page id of vector lane % 16 of tile t
    return btb[min((t * 16 + (lane_now() & 15)) / vpp, npages - 1)];
  };
  auto id_ok = [&](int id) { return id >= 0 && int64_t(id) < num_pages; };
  auto vec_off = [&](int t, int id) -> int64_t {
    const int x = t * 16 + (lane_now() & 15);
    return (int64_t(id_ok(id) ? id : 0) * Hkv + h) * D * P + (x % vpp) * TV;
  };
  auto shfl64 = [](int64_t v, int src) -> int64_t {
    const int l32 = __shfl(int(v), src, 64), h32 = __shfl(int(v >> 32), src, 64);
    return (int64_t(h32) << 32) | uint32_t(l32);
  };
  const int64_t P4 = 4 * int64_t(P), P16 = 16 * int64_t(P);
  auto load_k = [&](uint4 (&kr)[16], int64_t o, int i0) {
    const int l = lane_now(), kd = l >> 4, n16 = l & 15;
    const T* p = kpool + shfl64(o, n16) + (4 * i0 + kd) * int64_t(P);
#pragma unroll
    for (int i = 0; i < 16; ++i) kr[i] = tile32::load16<false>(p + i * P4);
  };
  auto load_v = [&](uint4 (&vr)[16], int64_t o, int u0) {
    const int l = lane_now(), kd = l >> 4, n16 = l & 15;
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const T* p = vpool + shfl64(o, 4 * kd + u0 + u) + n16 * int64_t(P);
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) vr[nb * NU + u] = tile32::load16<false>(p + nb * P16);
    }
  };

  float m = -INFINITY, lsum = 0.f;  // of row n16 (lsum: this lane's scores only)
  f32x4_t acc[NB];                  // rows 4 kd + j, column 16 nb + n16
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) acc[nb] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  if (wave < ntiles) {
    uint4 bufA[16], bufB[16];
    int t = wave;
    int bt_cur = load_bt(t), bt_nxt = load_bt(min(t + PR_WAVES, ntiles - 1));
    int64_t off_cur = vec_off(t, bt_cur);
    load_k(bufA, off_cur, 0);
    if constexpr (D == 128) load_k(bufB, off_cur, 16);
    else load_v(bufB, off_cur, 0);
    for (;;) {
      const bool has_next = t + PR_WAVES < ntiles;
      const int t_nxt = has_next ? t + PR_WAVES : t;
      const int bt_far = load_bt(min(t + 2 * PR_WAVES, ntiles - 1));
      // keys of vector n16 that some row of the item sees
      const int nv16 = id_ok(bt_cur) ? kmax - (t * 16 + (lane_now() & 15)) * TV : 0;
      const bool cut = __ballot(nv16 < TV) != 0;
      const bool edge = (t + 1) * TOK > kmin;  // rows of the item see different keys of the tile
      const int64_t off_nxt = vec_off(t_nxt, bt_nxt);

      f32x4_t s[TV];
#pragma unroll
      for (int c = 0; c < TV; ++c) s[c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      __builtin_amdgcn_sched_barrier(0);
      tile32::qk<DT>(bufA, &qs[lane_now() * QS], s);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (D == 128) {
        load_v(bufA, off_cur, 0);
        __builtin_amdgcn_sched_barrier(0);
        tile32::qk<DT>(bufB, &qs[lane_now() * QS + 16], s);
      } else {
        if (has_next) load_k(bufA, off_nxt, 0);
      }
      __builtin_amdgcn_sched_barrier(0);

      // softmax of row n16: token TV (4 kd + v) + c of the tile is s[c][v]
      if constexpr (DT != PIA_DTYPE_F32) {
#pragma unroll
        for (int c = 0; c < TV; ++c) s[c] *= scale_log2;
      }
      if (cut || edge) {
        const int kd = lane_now() >> 4;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int n = min(__shfl(nv16, 4 * kd + v, 64), lim - (t * 16 + 4 * kd + v) * TV);
#pragma unroll
          for (int c = 0; c < TV; ++c) s[c][v] = c < n ? s[c][v] : -INFINITY;
        }
      }
      float mx = -INFINITY;
#pragma unroll
      for (int c = 0; c < TV; ++c)
        mx = fmaxf(mx, fmaxf(fmaxf(s[c][0], s[c][1]), fmaxf(s[c][2], s[c][3])));
      const float mn = fmaxf(m, tile::max_col4(mx));
      // a row with no key yet: p = 2^-inf = 0
      const float nm = mn == -INFINITY ? 0.f : mn - tile32::kSplitShift<DT>;
      const bool moved = m != mn;
      const float alpha = moved ? __builtin_amdgcn_exp2f(m - mn) : 1.f;
      m = mn;
      float ps = 0.f;
#pragma unroll
      for (int c = 0; c < TV; ++c) {
#pragma unroll
        for (int v = 0; v < 4; ++v) s[c][v] = __builtin_amdgcn_exp2f(s[c][v] - nm);
        ps += (s[c][0] + s[c][1]) + (s[c][2] + s[c][3]);
      }
      lsum = lsum * alpha + ps;
      if (__ballot(moved)) {
        const int kd = lane_now() >> 4;
        float aj[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) aj[j] = __shfl(alpha, 4 * kd + j, 64);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[nb][j] *= aj[j];
      }

      // O += P . V over vectors u0 .. u0 + NU - 1
      auto pv_part = [&](uint4 (&vr)[16], int u0) {
        bool row_by_row = false;
        if (cut || edge) {
          const int kd = lane_now() >> 4;
          bool nf = false;
#pragma unroll
          for (int u = 0; u < NU; ++u) {
            const int n = __shfl(nv16, 4 * kd + u0 + u, 64);
            const int own = kmin - (t * 16 + 4 * kd + u0 + u) * TV;  // tokens every row sees
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
              uint4& x = vr[nb * NU + u];
              V::keep_below(x, n);
#pragma unroll
              for (int w = 0; w < 4; ++w) {
                const uint32_t bits = tile32::word(x, w);
                if constexpr (DT == PIA_DTYPE_F32)
                  nf |= w >= own && (bits & 0x7f800000u) == 0x7f800000u;
                else
                  nf |= (2 * w >= own && nonfinite16(bits, DT)) ||
                        (2 * w + 1 >= own && nonfinite16(bits >> 16, DT));
              }
            }
          }
          row_by_row = __ballot(nf) != 0;
        }
        if (!row_by_row) {
          tile32::pv<DT, NB, NU>(vr, s, u0, acc);
          return;
        }
        const int l = lane_now(), kd = l >> 4, n16 = l & 15;
#pragma unroll
        for (int u = 0; u < NU; ++u)
#pragma unroll
          for (int c = 0; c < TV; ++c)
            part[wave][n16 * TS + (NU * kd + u) * TV + c] = s[c][u0 + u];
        int lim_j[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) lim_j[j] = __shfl(lim, 4 * kd + j, 64);
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll 1
        for (int i = 0; i < 4 * NU * TV; ++i) {
          const int x = 4 * (i / TV / NU) + u0 + i / TV % NU, c = i % TV, tok = (t * 16 + x) * TV + c;
          if (c >= __builtin_amdgcn_readlane(nv16, x)) continue;
          const T* p = vpool + shfl64(off_cur, x) + c + n16 * int64_t(P);
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) {
            const float v = Elem<DT>::load(p, nb * P16);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const float pj = part[wave][(4 * kd + j) * TS + i];
              acc[nb][j] = tok < lim_j[j] ? fmaf(pj, v, acc[nb][j]) : acc[nb][j];
            }
          }
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
      };
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (D == 128) {
        load_v(bufB, off_cur, 2);
        __builtin_amdgcn_sched_barrier(0);
        pv_part(bufA, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (has_next) load_k(bufA, off_nxt, 0);
        __builtin_amdgcn_sched_barrier(0);
        pv_part(bufB, 2);
        __builtin_amdgcn_sched_barrier(0);
        if (has_next) load_k(bufB, off_nxt, 16);
      } else {
        pv_part(bufB, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (has_next) load_v(bufB, off_nxt, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (!has_next) break;
      t = t_nxt;
      bt_cur = bt_nxt;
      bt_nxt = bt_far;
      off_cur = off_nxt;
    }
  }

  // the waves' partials, then their merge: thread (row tid / 16, columns tid % 16 + 16 i)
  {
    const float l_row = tile32::sum_col4(lsum);
    const int kd = lane >> 4, n16 = lane & 15;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int j = 0; j < 4; ++j) part[wave][(4 * kd + j) * DS + 16 * nb + n16] = acc[nb][j];
    if (kd == 0) {
      part[wave][n16 * DS + D] = m;
      part[wave][n16 * DS + D + 1] = l_row;
    }
  }
  __syncthreads();
  const int r = tid >> 4, c16 = tid & 15, R = R0 + r;
  if (R >= n_rows) return;
  float M = -INFINITY, f[PR_WAVES], l = 0.f;
#pragma unroll
  for (int w = 0; w < PR_WAVES; ++w) M = fmaxf(M, part[w][r * DS + D]);
#pragma unroll
  for (int w = 0; w < PR_WAVES; ++w) {
    const float mw = part[w][r * DS + D];
    f[w] = mw == M ? 1.f : __builtin_amdgcn_exp2f(mw - M);
    l += part[w][r * DS + D + 1] * f[w];
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
  T* o = out + (row0 + R / G) * Hq * D + int64_t(h * G + R % G) * D;
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const int d = c16 + 16 * i;
    float a = 0.f;
#pragma unroll
    for (int w = 0; w < PR_WAVES; ++w) a += part[w][r * DS + d] * f[w];
    Elem<DT>::store(o, d, a * inv);
  }
}

template <int DT>
int launch_rows_dt(void* out, const void* q, const void* k_pages, const void* v_pages,
                   const int32_t* bt, int64_t bt_stride, const int32_t* kv_lens,
                   const int32_t* cu_q, const int32_t* offsets, int num_seqs,
                   int64_t total_q_rows, int Hq, int Hkv, int D, int P, int64_t num_pages,
                   float scale_log2, hipStream_t s) {
  using T = typename Elem<DT>::T;
  const int G = Hq / Hkv;
  // items: at most ceil(rows * G / 16) + one partial block per sequence, per kv head
  const int64_t items = (ceil_div(total_q_rows * G, PR_ROWS) + num_seqs) * Hkv;
  const dim3 grid{unsigned(ceil_div(items, 8) * 8), 1u, 1u};
#define PIA_PR(DD)                                                                             \
  hipLaunchKernelGGL((paged_attention_rows<DT, DD>), grid, dim3(64 * PR_WAVES), 0, s,          \
                     reinterpret_cast<T*>(out), reinterpret_cast<const T*>(q),                 \
                     reinterpret_cast<const T*>(k_pages), reinterpret_cast<const T*>(v_pages), \
                     bt, bt_stride, kv_lens, cu_q, offsets, num_seqs, int(total_q_rows), Hkv,  \
                     G, P, num_pages, scale_log2)
  if (D == 128) PIA_PR(128);
  else PIA_PR(64);
#undef PIA_PR
  return check_launch("paged_attention_rows");
}

}  // namespace

bool rows_path(int dtype, int Hq, int Hkv, int D, int P, int num_seqs, int64_t total_q_rows,
               const void* k_pages, const void* v_pages) {
  const int vec = dtype == PIA_DTYPE_F32 ? 4 : 8;
  const int64_t G = Hq / Hkv;
  // int32 row, item and workgroup counts
  const int64_t items = (ceil_div(total_q_rows * G, PR_ROWS) + num_seqs) * Hkv;
  return (D == 64 || D == 128) && P % vec == 0 && num_seqs <= PR_MAX_SEQS &&
         total_q_rows * G + PR_ROWS < (int64_t(1) << 31) && items + 8 < (int64_t(1) << 31) &&
         aligned(k_pages, 16) && aligned(v_pages, 16);
}

int launch_rows(int dtype, void* out, const void* q, const void* k_pages, const void* v_pages,
                const int32_t* bt, int64_t bt_stride, const int32_t* kv_lens,
                const int32_t* cu_q, const int32_t* offsets, int num_seqs, int64_t total_q_rows,
                int Hq, int Hkv, int D, int P, int64_t num_pages, float scale_log2,
                hipStream_t s) {
  auto* launch = dtype == PIA_DTYPE_F32   ? &launch_rows_dt<PIA_DTYPE_F32>
                 : dtype == PIA_DTYPE_F16 ? &launch_rows_dt<PIA_DTYPE_F16>
                                          : &launch_rows_dt<PIA_DTYPE_BF16>;
  return launch(out, q, k_pages, v_pages, bt, bt_stride, kv_lens, cu_q, offsets, num_seqs,
                total_q_rows, Hq, Hkv, D, P, num_pages, scale_log2, s);
}

}  // namespace pia
