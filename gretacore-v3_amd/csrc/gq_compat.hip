// gq_compat.hip -- the reference's INT8 / INT4 weight-only launchers, with the
// same arguments, for callers that keep the reference's requantized weight
// formats (weight_loader.cpp:668-1008):
//   launch_gemm_mfma_int8_wt_fp32_acc32  gemm_kernels.hip:742-760
//   launch_gemm_mfma_int4_wt_fp32_acc32  gemm_kernels.hip:910-942
// Semantics: c[m][n] = (sum_k a[m][k] * (w[n][k] * s[idx(n, k)])) * h[n/hd]
// with fp32 accumulation, written in the mathematical ("row") layout
// c[m*ldc + n].  Rows of a are lda apart.  M, N or K == 0 returns at once.
//
// Up to 32 rows (and with force_gemv) the GEMV in fp32, as the reference's
// GEMV kernels -- on the VALU for small calls, on the matrix cores with fp32
// precision (k_compat_mfma) for more; above, the reference's MFMA route on fp16 operands through
// gq_gemm (compat_gemm_route).
#include "gq_internal.h"

namespace {

// Scale of weight (n, k).  The reference's two routes index the per-group
// scales differently: its GEMV kernels (M <= 32 or force_gemv) take
// s_row = scales + (n*K)/gs and s_row[k/gs] (gemm_kernels.hip:610,615 and
// 781,796-797), its MFMA kernels (M > 32) scales[(n*K + k)/gs]
// (gemm_kernels.hip:717, 886).  srow selects the first form; the two agree
// whenever K % gs == 0.
GQ_DEV size_t scale_idx(size_t n, size_t K, size_t k, int gs, int srow) {
  return srow ? (n * K) / (size_t)gs + k / (size_t)gs : (n * K + k) / (size_t)gs;
}
// The same with the row's part computed once: for row n, q0 = (n K) / gs and
// r0 = (n K) % gs; a lane's index for k is then q0 + k / gs (srow) or
// q0 + (r0 + k) / gs, one 32-bit division -- a shift where gs is a power of
// two (gsh >= 0) -- instead of a 64-bit division per load.
struct RowScale {
  size_t q0;
  uint32_t r0;
};
GQ_DEV RowScale row_scale(size_t n, size_t K, int gs) {
  const size_t nk = n * K;
  return RowScale{nk / (size_t)gs, (uint32_t)(nk % (size_t)gs)};
}
GQ_DEV int gs_shift(int gs) { return (gs & (gs - 1)) == 0 ? __builtin_ctz((unsigned)gs) : -1; }
GQ_DEV size_t scale_idx_row(RowScale rsc, uint32_t k, int gs, int gsh, int srow) {
  const uint32_t x = srow ? k : rsc.r0 + k;
  return rsc.q0 + (gsh >= 0 ? x >> gsh : x / (uint32_t)gs);
}

GQ_DEV float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

template <typename TA>
GQ_DEV float ld_a(const TA *p) { return (float)*p; }

template <int MB, typename TA, bool INT4>
__global__ void __launch_bounds__(256)
k_compat_gemv(const TA *__restrict__ a, const uint8_t *__restrict__ b, float *__restrict__ c,
              const float *__restrict__ scales, const float *__restrict__ head_scales, int M, int N, int K,
              int lda, int ldc, int gs, int srow, int head_dim, int m_base) {
  const int lane = threadIdx.x & 63;
  const int n = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (n >= N) return;
  const int mcount = min(MB, M - m_base);
  float acc[MB];
#pragma unroll
  for (int i = 0; i < MB; ++i) acc[i] = 0.f;
  const size_t row_elems = (size_t)n * K;
  // lane covers 16 consecutive k per step; the wave covers 1024 k per step
  for (int k0 = lane * 16; k0 < K; k0 += 1024) {
    float wv[16];
    if (k0 + 16 <= K && (K % 16) == 0) {
      if constexpr (INT4) {
        gq_u2 p = gq_ld8(b + (row_elems + k0) / 2);
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          uint32_t byte = (p[e >> 3] >> (8 * ((e >> 1) & 3))) & 0xFFu;
          int v = (e & 1) ? (int)(byte >> 4) : (int)(byte & 15u);
          v = (v ^ 8) - 8;
          wv[e] = (float)v;
        }
      } else {
        gq_u4 p = gq_ld16(b + row_elems + k0);
#pragma unroll
        for (int e = 0; e < 16; ++e) wv[e] = (float)(int8_t)((p[e >> 2] >> (8 * (e & 3))) & 0xFFu);
      }
#pragma unroll
      for (int e = 0; e < 16; ++e) wv[e] = wv[e] * (scales ? scales[scale_idx(n, K, k0 + e, gs, srow)] : 1.0f);
    } else {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        int k = k0 + e;
        float v = 0.f;
        if (k < K) {
          size_t idx = row_elems + k;
          int q;
          if constexpr (INT4) {
            uint32_t byte = b[idx / 2];
            q = (idx & 1) ? (int)(byte >> 4) : (int)(byte & 15u);
            q = (q ^ 8) - 8;
          } else {
            q = (int8_t)b[idx];
          }
          v = (float)q * (scales ? scales[scale_idx(n, K, k, gs, srow)] : 1.0f);
        }
        wv[e] = v;
      }
    }
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      if (i >= mcount) break;
      const TA *ar = a + (size_t)(m_base + i) * lda;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        int k = k0 + e;
        float x = k < K ? ld_a(ar + k) : 0.f;
        acc[i] += x * wv[e];
      }
    }
  }
  float h = (head_scales && head_dim > 0) ? head_scales[n / head_dim] : 1.0f;
#pragma unroll
  for (int i = 0; i < MB; ++i) {
    if (i >= mcount) break;
    float s = wave_sum(acc[i]);
    if (lane == 0) c[(size_t)(m_base + i) * ldc + n] = s * h;
  }
}

// Streaming form for K % 16 == 0 and group sizes that are multiples of 16 (a
// lane's 16 k then share one scale): a wave takes RW = 4 rows and walks K in
// 1024-k segments, 16 k per lane; per segment it loads the MB activation rows'
// 16 values once (float4 loads) for all its rows, each row's 16 weights with
// one 16- (INT8) or 8-byte (INT4) load and one scale, and accumulates
// s * sum(q * x) in fp32.  The sum over a lane's 16 terms is then scaled once
// where the reference scales each weight: the result differs only by fp32
// rounding order.
template <int MB, int RW, typename TA, bool INT4>
__global__ void __launch_bounds__(256)
k_compat_gemv_seg(const TA *__restrict__ a, const uint8_t *__restrict__ b, float *__restrict__ c,
                  const float *__restrict__ scales, const float *__restrict__ head_scales, int M, int N, int K,
                  int lda, int ldc, int gs, int srow, int head_dim) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = ((int)blockIdx.x * 4 + wave) * RW;
  if (n0 >= N) return;
  const int m_base = (int)blockIdx.y * MB;
  const int mcount = min(MB, M - m_base);
  float acc[RW][MB];
#pragma unroll
  for (int r = 0; r < RW; ++r)
#pragma unroll
    for (int i = 0; i < MB; ++i) acc[r][i] = 0.f;
  const TA *arow[MB];
#pragma unroll
  for (int i = 0; i < MB; ++i) arow[i] = a + (size_t)(m_base + (i < mcount ? i : 0)) * lda;
  const int gsh = gs_shift(gs);
  RowScale rsc[RW];
#pragma unroll
  for (int r = 0; r < RW; ++r) rsc[r] = row_scale((size_t)(n0 + r < N ? n0 + r : N - 1), (size_t)K, gs);
#pragma unroll 2
  for (int k0 = 16 * lane; k0 < K; k0 += 1024) {
    float xv[MB][16];
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      if constexpr (sizeof(TA) == 4) {
        const gq_f4 *p = reinterpret_cast<const gq_f4 *>(reinterpret_cast<const float *>(arow[i]) + k0);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const gq_f4 v = p[q];
          xv[i][4 * q] = v[0];
          xv[i][4 * q + 1] = v[1];
          xv[i][4 * q + 2] = v[2];
          xv[i][4 * q + 3] = v[3];
        }
      } else {
        const gq_half8 *p = reinterpret_cast<const gq_half8 *>(reinterpret_cast<const _Float16 *>(arow[i]) + k0);
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const gq_half8 v = p[q];
#pragma unroll
          for (int e = 0; e < 8; ++e) xv[i][8 * q + e] = (float)v[e];
        }
      }
    }
#pragma unroll
    for (int r = 0; r < RW; ++r) {
      const int n = n0 + r < N ? n0 + r : N - 1;  // (rows past N are computed, never stored)
      const size_t idx = (size_t)n * K + k0;
      float wv[16];
      if constexpr (INT4) {
        const gq_u2 p = gq_ld8(b + idx / 2);
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const uint32_t byte = (p[e >> 3] >> (8 * ((e >> 1) & 3))) & 0xFFu;
          const int v = (int)((e & 1) ? (byte >> 4) : (byte & 15u));
          wv[e] = (float)((v ^ 8) - 8);
        }
      } else {
        const gq_u4 p = gq_ld16(b + idx);
#pragma unroll
        for (int e = 0; e < 16; ++e) wv[e] = (float)(int8_t)((p[e >> 2] >> (8 * (e & 3))) & 0xFFu);
      }
      const float sc = scales ? scales[scale_idx_row(rsc[r], (uint32_t)k0, gs, gsh, srow)] : 1.0f;
#pragma unroll
      for (int i = 0; i < MB; ++i) {
        float d = 0.f;
#pragma unroll
        for (int e = 0; e < 16; ++e) d += xv[i][e] * wv[e];
        acc[r][i] += sc * d;
      }
    }
  }
#pragma unroll
  for (int r = 0; r < RW; ++r) {
    const int n = n0 + r;
    const float h = (head_scales && head_dim > 0 && n < N) ? head_scales[n / head_dim] : 1.0f;
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      const float sum = wave_sum(acc[r][i]);
      if (lane == 0 && n < N && i < mcount) c[(size_t)(m_base + i) * ldc + n] = sum * h;
    }
  }
}

// One-row-per-wave form with the activations in LDS (fp32, all of K for MB
// rows, staged once per workgroup of 16 waves): the activation traffic per
// workgroup is K * MB * 4 bytes for 16 rows instead of per wave.  Each lane
// takes 16 k per 1024-k segment; its weights for all segments are requested
// up front (at most NSEG segments).  The LDS holds 16-byte chunks at
// c ^ ((c >> 4) & 3) so the four 16-byte reads of a lane's 16 values hit 16
// different bank groups across each 16 lanes.
template <int MB, int NSEG, typename TA, bool INT4, int RW = 1>
__global__ void __launch_bounds__(1024)
k_compat_gemv_lds(const TA *__restrict__ a, const uint8_t *__restrict__ b, float *__restrict__ c,
                  const float *__restrict__ scales, const float *__restrict__ head_scales, int M, int N, int K,
                  int lda, int ldc, int gs, int srow, int head_dim) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  gq_f4 *xs = reinterpret_cast<gq_f4 *>(lds_raw);  // [MB][K / 4] chunks, swizzled
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int m_base = (int)blockIdx.y * MB;
  const int mcount = min(MB, M - m_base);
  const int n0 = ((int)blockIdx.x * 16 + __builtin_amdgcn_readfirstlane(wave)) * RW;
  const int nseg = (K + 1023) / 1024;
  const int gsh = gs_shift(gs);
  // weights and scales of every segment of the wave's RW rows first (clamped,
  // unconditional; a row past N is computed, never stored)
  gq_u4 w8[RW][INT4 ? 1 : NSEG];
  gq_u2 w4[RW][INT4 ? NSEG : 1];
  float sc[RW][NSEG];
#pragma unroll
  for (int r = 0; r < RW; ++r) {
    const int nr = n0 + r < N ? n0 + r : N - 1;
    const RowScale rsc = row_scale((size_t)nr, (size_t)K, gs);
#pragma unroll
    for (int it = 0; it < NSEG; ++it) {
      int k0 = 16 * lane + 1024 * it;
      k0 = k0 < K ? k0 : K - 16;
      const size_t idx = (size_t)nr * K + k0;
      if constexpr (INT4) w4[r][it] = gq_ld8(b + idx / 2);
      else w8[r][it] = gq_ld16(b + idx);
      sc[r][it] = scales ? scales[scale_idx_row(rsc, (uint32_t)k0, gs, gsh, srow)] : 1.0f;
    }
  }
  // activations -> LDS
  const int nchunk = K / 4;
  for (int i = (int)threadIdx.x; i < MB * nchunk; i += 1024) {
    const int row = i / nchunk, ch = i % nchunk;
    gq_f4 v = gq_f4{0.f, 0.f, 0.f, 0.f};
    if (row < mcount) {
      const TA *src = a + (size_t)(m_base + row) * lda + 4 * ch;
      if constexpr (sizeof(TA) == 4) {
        v = *reinterpret_cast<const gq_f4 *>(src);
      } else {
        const _Float16 *h = reinterpret_cast<const _Float16 *>(src);
        v = gq_f4{(float)h[0], (float)h[1], (float)h[2], (float)h[3]};
      }
    }
    xs[row * nchunk + (ch ^ ((ch >> 4) & 3))] = v;
  }
  __syncthreads();
  float acc[RW][MB];
#pragma unroll
  for (int r = 0; r < RW; ++r)
#pragma unroll
    for (int i = 0; i < MB; ++i) acc[r][i] = 0.f;
#pragma unroll
  for (int it = 0; it < NSEG; ++it) {
    const int k0 = 16 * lane + 1024 * it;
    if (it < nseg && k0 < K) {
      float xv[MB][16];
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int ch = k0 / 4 + j;
          const gq_f4 x4 = xs[i * nchunk + (ch ^ ((ch >> 4) & 3))];
          xv[i][4 * j] = x4[0];
          xv[i][4 * j + 1] = x4[1];
          xv[i][4 * j + 2] = x4[2];
          xv[i][4 * j + 3] = x4[3];
        }
#pragma unroll
      for (int r = 0; r < RW; ++r) {
        float wv[16];
        if constexpr (INT4) {
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            const uint32_t byte = (w4[r][it][e >> 3] >> (8 * ((e >> 1) & 3))) & 0xFFu;
            const int v = (int)((e & 1) ? (byte >> 4) : (byte & 15u));
            wv[e] = (float)((v ^ 8) - 8);
          }
        } else {
#pragma unroll
          for (int e = 0; e < 16; ++e) wv[e] = (float)(int8_t)((w8[r][it][e >> 2] >> (8 * (e & 3))) & 0xFFu);
        }
#pragma unroll
        for (int i = 0; i < MB; ++i) {
          float d = 0.f;
#pragma unroll
          for (int e = 0; e < 16; ++e) d += xv[i][e] * wv[e];
          acc[r][i] += sc[r][it] * d;
        }
      }
    }
  }
#pragma unroll
  for (int r = 0; r < RW; ++r) {
    const int n = n0 + r;
    const float h = (head_scales && head_dim > 0 && n < N) ? head_scales[n / head_dim] : 1.0f;
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      const float sum = wave_sum(acc[r][i]);
      if (lane == 0 && n < N && i < mcount) c[(size_t)(m_base + i) * ldc + n] = sum * h;
    }
  }
}

// ---- matrix-core form: 3..32 rows (any count with force_gemv) -----------------
// The codes against the activations with nothing of either lost on the way to the
// products; fp32 sums.
//  - fp32 activations: three bf16 limbs, x = hi + mid + lo, each the top 8 bits of what
//    is left: 24 bits at any exponent (the codes are exact in bf16).  The MFMA takes
//    subnormal inputs as zeros, so a row's window below 2^-60 goes in times 2^66; entries
//    under 2^-110 beside one above 2^-63 keep their first 8 or 16 bits.
//    (Two fp16 limbs under one power of two per 256 k kept 22 bits of a window's
//    largest entries and fewer of the rest: with an entry 1e7 times the others, whose
//    code was 0, 9e-5 off.  v_mfma_f32_16x16x4_f32 instead, 1/16 of the rate: 8 rows
//    of 14336 x 4096, INT4, 29 us; v_mfma_f32_4x4x1 with its 16 blocks 24.5.)
//  - fp16 activations: as they are (the codes are exact in fp16).
// v_mfma_f32_16x16x32 is one scale group of 32 for 16 weight rows and 16 activation
// rows; the limbs go to one fp32 accumulator, lowest first, which is scaled by the
// group's factor and added to the window's sum, that to the total, compensated.
// Up to 8 rows two MFMAs do: A rows 0..7 hold hi and 8..15 mid, then lo / 2 both
// times, and the two halves of D are added at the end.  Odd groups count the
// codes negated and with -s: the MFMA's internal sum rounds downwards, a bias that
// would otherwise add up over K.
//
// What bounds it is VALU work: a code's way to bf16 (v_cvt_off_f32_i4 or a byte's
// conversion, and half a packing) and the limbs' making.  14336 x 4096, INT4 / INT8,
// VALU kernels -> this: 8 rows 44 / 51 -> 19.1 / 23.6 us, 32 rows 155 / 172 -> 31 / 36;
// rel-L2 against float64 8.9e-8 at 8 rows (VALU kernels 1.1-1.2e-7).
//
// Workgroup: TW row tiles of 16 x KS parts of K, one wave each.  The operands of
// a window (WIN k of every part) are made once per workgroup in LDS, double-
// buffered where that fits; a wave's 16-byte weight loads (lane (g, r): row r, 16-byte
// piece g of 64) go out two windows ahead.  A piece is one group's (INT4) or half a
// group's (INT8) codes of one row, so lane swaps (permlane) turn four pieces into
// B fragments of one group each; k order inside a group is free as long as the
// activations are stored alike.
template <bool INT4>
struct CmGroup {  // 128 k of 16 rows: four groups' codes and scales
  gq_u4 q[INT4 ? 1 : 2];
  float s;  // lane (g, r): the scale of group g of row r
};

// lane groups (g0 g1 g2 g3) of a and b -> a: (a0 a1 b0 b1), b: (a2 a3 b2 b3)
GQ_DEV void cm_swap32(uint32_t &a, uint32_t &b) {
  const auto v = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = v[0];
  b = v[1];
}
// -> a: (a0 b0 a2 b2), b: (a1 b1 a3 b3)
GQ_DEV void cm_swap16(uint32_t &a, uint32_t &b) {
  const auto v = __builtin_amdgcn_permlane16_swap(a, b, false, false);
  a = v[0];
  b = v[1];
}

typedef __bf16 cm_bf8 __attribute__((ext_vector_type(8)));
typedef __bf16 cm_bf2 __attribute__((ext_vector_type(2)));

GQ_DEV uint32_t cm_max_row(uint32_t v) {  // largest of each 16 lanes (DPP; 0 is max's identity)
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, true));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xF, 0xF, true));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xF, 0xF, true));
  return max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x140, 0xF, 0xF, true));
}

template <bool INT4, typename TA, int MR, int WIN, int TW, int KS>
__global__ void __launch_bounds__(64 * TW * KS, MR == 32 && KS == 2 ? 4 : 1)
k_compat_mfma(const TA *__restrict__ a, const uint8_t *__restrict__ b, float *__restrict__ c,
              const float *__restrict__ scales, const float *__restrict__ head_scales, int M, int N, int K, int lda,
              int ldc, int head_dim, int NI) {
  // K part blockIdx.z of gridDim.z: its windows, its own M x N of c
  const int z0 = (K + WIN - 1) / WIN * (int)blockIdx.z / (int)gridDim.z;
  const int nw = (K + WIN - 1) / WIN * ((int)blockIdx.z + 1) / (int)gridDim.z - z0;
  c += (size_t)blockIdx.z * (size_t)M * (size_t)ldc;
  constexpr bool F32 = sizeof(TA) == 4;
  static_assert(F32 || INT4, "fp16 activations: INT4 only");
  constexpr int U = F32 ? 3 : 1;              // limbs
  constexpr int NG = WIN / 128;               // 128-k groups per window
  constexpr int NB = WIN / 32;                // scale groups per window
  constexpr int RUN = WIN / 8;                // runs of 8 per row and window
  constexpr int NT = 64 * TW * KS;
  constexpr int RPT = KS * MR * RUN / NT;     // runs per thread and window
  constexpr int MT = MR > 16 ? MR / 16 : 1;   // 16-row tiles of activations
  constexpr int WB = NB * U * 4 * MR * 16;    // LDS bytes of a part's window: [NB][U][4][MR][16]
  static_assert(RPT >= 1 && RPT * NT == KS * MR * RUN && (RUN == 16 || RUN == 32), "runs divide evenly");
  // buffers: two where they leave room for the workgroups a CU should hold (16 waves)
  constexpr int XB = 2 * KS * WB <= (TW * KS > 8 ? 160 : 80) * 1024 ? 2 : 1;
  __shared__ __attribute__((aligned(16))) unsigned char xs[XB][KS][WB];
  __shared__ __attribute__((aligned(16))) float xsc[XB][KS * MR];  // what a part's row of the window counts for
  static_assert(sizeof(xs) >= (size_t)KS * TW * MT * 64 * 16, "the parts' sums reuse it");
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tt = wave % TW, part = wave / TW;
  const int g = lane >> 4, r = lane & 15;
  const int m_base = (int)blockIdx.y * MR;
  const int nb = K / 32;
  const int w0 = z0 + nw * part / KS, w1 = z0 + nw * (part + 1) / KS;  // this wave's windows (<= NI)
  const int n = ((int)blockIdx.x * TW + tt) * 16 + r;
  const int nr = n < N ? n : N - 1;  // (rows past N are computed, never stored)
  const uint8_t *wrow = b + (size_t)nr * K / (INT4 ? 2 : 1);
  const float *srow = scales + (size_t)nr * nb;

  // weights and scales of window w; past the row's end another group's are
  // read instead, with scale 0 (their activations are zeros too)
  auto load_win = [&](int w, CmGroup<INT4> (&gr)[NG]) {
    w = w < w1 ? w : w1 - 1;
#pragma unroll
    for (int j = 0; j < NG; ++j) {
      const int b0 = w * NB + 4 * j;
      if constexpr (INT4) {
        const int bi = b0 + g < nb ? b0 + g : nb - 1;
        gr[j].q[0] = gq_ld16(wrow + 16 * (size_t)bi);
      } else {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int bi = b0 + 2 * h + (g >> 1) < nb ? b0 + 2 * h + (g >> 1) : nb - 1;
          gr[j].q[h] = gq_ld16(wrow + 32 * (size_t)bi + 16 * (g & 1));
        }
      }
      const float s = srow[b0 + g < nb ? b0 + g : nb - 1];
      gr[j].s = b0 + g < nb ? s : 0.f;
    }
  };
  // activations: run u of this thread = (part, row, run of the window)
  constexpr int XU = F32 ? 2 : 1;  // 16-byte loads of a run
  gq_u4 xv[RPT][XU];
  auto load_x = [&](int it) {
#pragma unroll
    for (int u = 0; u < RPT; ++u) {
      const int run = (int)threadIdx.x + u * NT;
      const int kr = run % RUN, row = (run / RUN) % MR, p = run / (RUN * MR);
      const int w = z0 + nw * p / KS + it;
      const int k = w * WIN + 8 * kr;
      const bool in = m_base + row < M && w < z0 + nw * (p + 1) / KS && k < K;  // (K % 32 == 0: a run is whole)
      const gq_u4 *src = reinterpret_cast<const gq_u4 *>(a + (size_t)(in ? m_base + row : 0) * lda + (in ? k : 0));
#pragma unroll
      for (int i = 0; i < XU; ++i) {
        const gq_u4 v = src[i];
#pragma unroll
        for (int e = 0; e < 4; ++e) xv[u][i][e] = in ? v[e] : 0u;
      }
    }
  };
  // A limb's units of a group: [4 lane groups][rows][16].  The row's place is
  // exclusive-or'ed with the unit's, so the runs that consecutive lanes store lie in
  // different banks.  Limbs (offsets from the group's): MR = 8: 16 rows hi and
  // mid, 8 rows lo / 2; else one after the other
  constexpr int GB = U * 4 * MR * 16;                  // bytes of a group
  constexpr int R0 = F32 && MR == 8 ? 16 : MR;         // rows of the first unit
  constexpr int MID = MR == 8 ? 8 * 16 : 4 * MR * 16;  // hi -> mid
  auto store_x = [&](int buf) {
#pragma unroll
    for (int u = 0; u < RPT; ++u) {
      const int run = (int)threadIdx.x + u * NT;
      const int kr = run % RUN, row = (run / RUN) % MR, p = run / (RUN * MR);
      const int blk = kr >> 2, unit = kr & 3;
      const int gq = INT4 ? unit : ((unit & 1) << 1) | (unit >> 1);  // (the INT8 swap's order)
      const int rx = row ^ (gq | (blk & 1) << 2);
      unsigned char *d = &xs[XB == 2 ? buf : 0][p][blk * GB + (gq * R0 + rx) * 16];
      if constexpr (F32) {
        float x[8], m[8], l[8], t = 0.f, us = 1.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          x[e] = __uint_as_float(xv[u][e >> 2][e & 3]);
          t += fabsf(x[e]);
        }
        const bool odd = t != 0.f && !(t >= 0x1p-60f && t < __builtin_inff());  // small or not finite
        const bool any = __any(odd);
        if (any) {
          float mx = 0.f;
#pragma unroll
          for (int e = 0; e < 8; ++e) mx = fmaxf(mx, fabsf(x[e]));
          uint32_t wm = cm_max_row(__float_as_uint(mx));  // (the window's RUN lanes are consecutive)
          if constexpr (RUN == 32) {
            const auto v = __builtin_amdgcn_permlane16_swap(wm, wm, false, false);
            wm = max(v[0], v[1]);
          }
          const bool up = __uint_as_float(wm) < 0x1p-60f;
          us = up ? 0x1p-66f : 1.f;
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            x[e] *= up ? 0x1p66f : 1.f;
            if (x[e] != x[e]) x[e] = __uint_as_float(0x7FC00000u);
          }
        }
        if (kr == 0) xsc[XB == 2 ? buf : 0][p * MR + row] = us * (INT4 ? 16.f : 1.f);  // (INT4 codes: by sixteenths)
#pragma unroll
        for (int e = 0; e < 8; ++e) m[e] = x[e] - __uint_as_float(__float_as_uint(x[e]) & 0xFFFF0000u);
        if (any) {  // (an Inf or NaN is its first limb alone)
#pragma unroll
          for (int e = 0; e < 8; ++e) m[e] = fabsf(x[e]) < __builtin_inff() ? m[e] : 0.f;
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          l[e] = m[e] - __uint_as_float(__float_as_uint(m[e]) & 0xFFFF0000u);
          if constexpr (MR == 8) l[e] *= 0.5f;
        }
        auto put = [&](unsigned char *to, const float (&v)[8]) {
          gq_u4 o;
#pragma unroll
          for (int e = 0; e < 4; ++e)  // (the upper halves of two)
            o[e] = __builtin_amdgcn_perm(__float_as_uint(v[2 * e + 1]), __float_as_uint(v[2 * e]), 0x07060302u);
          *reinterpret_cast<gq_u4 *>(to) = o;
        };
        put(d, x);
        put(d + MID, m);
        put(MR == 8 ? &xs[XB == 2 ? buf : 0][p][blk * GB + (4 * 16 + gq * 8 + rx) * 16] : d + 2 * MID, l);
      } else {
        // (the order of gq_nib_halves over plain nibbles: k 0 4 1 5 2 6 3 7)
        const uint32_t x0 = xv[u][0][0], x1 = xv[u][0][1], x2 = xv[u][0][2], x3 = xv[u][0][3];
        *reinterpret_cast<gq_u4 *>(d) =
            gq_u4{__builtin_amdgcn_perm(x2, x0, 0x05040100u), __builtin_amdgcn_perm(x2, x0, 0x07060302u),
                  __builtin_amdgcn_perm(x3, x1, 0x05040100u), __builtin_amdgcn_perm(x3, x1, 0x07060302u)};
      }
    }
  };

  // (comp: what rounding took from the windows' sum so far)
  gq_f4 acc[MT], comp[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = comp[t] = gq_f4{0.f, 0.f, 0.f, 0.f};
  const uint32_t mg = gq_nib_magic();
  // the lane's A row in an even and an odd group's units
  const int r8 = MR == 8 ? (r & 7) : r;
  const int ra = F32 ? r : r8;  // (the first unit's row)
  const int xo[2] = {(g * R0 + (ra ^ g)) * 16, (g * R0 + (ra ^ (g | 4))) * 16};
  const int xl[2] = {(64 + g * 8 + (r8 ^ g)) * 16, (64 + g * 8 + (r8 ^ (g | 4))) * 16};  // (MR = 8: lo / 2)
  auto consume = [&](int it, CmGroup<INT4> (&gr)[NG]) {
    if (w0 + it >= w1) return;
    const unsigned char *xb = xs[XB == 2 ? it & 1 : 0][part];
    gq_f4 wa[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) wa[t] = gq_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < NG; ++j) {
      // scales of the four groups, each for every lane group
      uint32_t sv[4];
      sv[0] = sv[2] = __float_as_uint(gr[j].s);
      cm_swap32(sv[0], sv[2]);
      sv[1] = sv[0];
      sv[3] = sv[2];
      cm_swap16(sv[0], sv[1]);
      cm_swap16(sv[2], sv[3]);
      // lane group g: codes 8 g .. 8 g + 7 of each group (INT8: in the swap's order)
      uint32_t q[4][INT4 ? 1 : 2];
      if constexpr (INT4) {
#pragma unroll
        for (int e = 0; e < 4; ++e) q[e][0] = gr[j].q[0][e];
        cm_swap32(q[0][0], q[2][0]);
        cm_swap32(q[1][0], q[3][0]);
        cm_swap16(q[0][0], q[1][0]);
        cm_swap16(q[2][0], q[3][0]);
      } else {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            q[2 * h][e] = gr[j].q[h][e];
            q[2 * h + 1][e] = gr[j].q[h][2 + e];
            cm_swap32(q[2 * h][e], q[2 * h + 1][e]);
          }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const unsigned char *xg = xb + (4 * j + i) * GB + xo[i & 1];
        const float s = (i & 1) ? -__uint_as_float(sv[i]) : __uint_as_float(sv[i]);
        gq_f4 d[MT];
        if constexpr (F32) {
          cm_bf8 bf;
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            float f;
            if constexpr (INT4) f = __builtin_amdgcn_cvt_off_f32_i4((int)(q[i][0] >> (4 * e)));  // code / 16
            else f = (float)(int8_t)(q[i][e >> 2] >> (8 * (e & 3)));
            bf[e] = (__bf16)((i & 1) ? -f : f);
          }
          auto rd = [&](const unsigned char *at) { return *reinterpret_cast<const cm_bf8 *>(at); };
#pragma unroll
          for (int t = 0; t < MT; ++t) {
            const gq_f4 z = gq_f4{0.f, 0.f, 0.f, 0.f};
            if constexpr (MR == 8) {
              d[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(rd(xb + (4 * j + i) * GB + xl[i & 1]), bf, z, 0, 0, 0);
            } else {
              d[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(rd(xg + 2 * MID + 256 * t), bf, z, 0, 0, 0);
              d[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(rd(xg + MID + 256 * t), bf, d[t], 0, 0, 0);
            }
            d[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(rd(xg + 256 * t), bf, d[t], 0, 0, 0);
          }
        } else {
          gq_half2 p[4];
          // (1024 + u, 1024 + 16 u) -> u - 8, u = code + 8
          gq_nib_halves(q[i][0] ^ 0x88888888u, mg, p);
          const gq_half2 b1 = {(_Float16)-1032.f, (_Float16)-1032.f}, b16 = {(_Float16)-72.f, (_Float16)-72.f};
          const gq_half2 k16 = {(_Float16)0.0625f, (_Float16)0.0625f};
          gq_half8 bf;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const gq_half2 v = (e & 1) ? __builtin_elementwise_fma(p[e], k16, b16) : p[e] + b1;
            bf[2 * e] = (i & 1) ? -v[0] : v[0];
            bf[2 * e + 1] = (i & 1) ? -v[1] : v[1];
          }
#pragma unroll
          for (int t = 0; t < MT; ++t)
            d[t] = gq_mfma16(*reinterpret_cast<const gq_half8 *>(xg + 256 * t), bf, gq_f4{0.f, 0.f, 0.f, 0.f});
        }
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
          for (int v = 0; v < 4; ++v) wa[t][v] = fmaf(s, d[t][v], wa[t][v]);
      }
    }
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      gq_f4 us = gq_f4{1.f, 1.f, 1.f, 1.f};
      if constexpr (F32)
        us = *reinterpret_cast<const gq_f4 *>(&xsc[XB == 2 ? it & 1 : 0][part * MR + 16 * t + ((4 * g) & (MR - 1) & 15)]);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float y = fmaf(wa[t][v], us[v], -comp[t][v]), z = acc[t][v] + y;
        comp[t][v] = fabsf(z) < __builtin_inff() ? (z - acc[t][v]) - y : 0.f;  // (an Inf stays one)
        acc[t][v] = z;
      }
    }
  };

  // the weights of the next two windows and the activations of the next one are
  // requested before a window is consumed; three weight buffers rotate by
  // unrolling (no load under a branch: surplus ones re-read the last window)
  CmGroup<INT4> b0[NG], b1[NG], b2[NG];
  load_x(0);
  load_win(w0, b0);
  load_win(w0 + 1, b1);
  store_x(0);
  __syncthreads();
  auto window = [&](int it, CmGroup<INT4> (&cur)[NG], CmGroup<INT4> (&nxt)[NG]) {
    load_x(it + 1);
    load_win(w0 + it + 2, nxt);
    consume(it, cur);
    if constexpr (XB == 1) __syncthreads();  // (every wave has read the window)
    store_x((it + 1) & 1);
    __syncthreads();
  };
  for (int it = 0; it < NI; it += 3) {
    window(it, b0, b2);
    if (it + 1 >= NI) break;
    window(it + 1, b1, b0);
    if (it + 2 >= NI) break;
    window(it + 2, b2, b1);
  }
  if constexpr (F32 && MR == 8) {  // (D rows 8..15, lane groups 2 and 3: the mid limbs' of rows 0..7)
#pragma unroll
    for (int v = 0; v < 4; ++v) acc[0][v] += __shfl_xor(acc[0][v], 32, 64);
  }
  // the parts' sums through LDS, added in part order
  gq_f4 *red = reinterpret_cast<gq_f4 *>(&xs[0][0][0]);  // [KS][TW][MT][64]
#pragma unroll
  for (int t = 0; t < MT; ++t) red[((part * TW + tt) * MT + t) * 64 + lane] = acc[t];
  __syncthreads();
  if (part != 0 || n >= N) return;
  const float h = (head_scales && head_dim > 0) ? head_scales[n / head_dim] : 1.0f;
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    gq_f4 sum = acc[t];
#pragma unroll
    for (int p = 1; p < KS; ++p) {
      const gq_f4 v = red[((p * TW + tt) * MT + t) * 64 + lane];
#pragma unroll
      for (int e = 0; e < 4; ++e) sum[e] += v[e];
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int row = 16 * t + 4 * g + v;  // D row (MR = 8: rows 8..15 repeat 0..7)
      if (row < MR && m_base + row < M) c[(size_t)(m_base + row) * ldc + n] = sum[v] * h;
    }
  }
}

// c = h * (the K parts' sums [parts][M][N] added in part order, compensated)
__global__ void __launch_bounds__(256) k_cm_sum(const float *__restrict__ part, const float *__restrict__ head_scales,
                                                float *__restrict__ c, int M, int N, int ldc, int head_dim, int parts) {
  const int n = (int)blockIdx.x * 256 + (int)threadIdx.x, m = (int)blockIdx.y;
  if (n >= N) return;
  const size_t mn = (size_t)M * N, i = (size_t)m * N + n;
  float sum = part[i], comp = 0.f;
  for (int p = 1; p < parts; ++p) {
    const float y = part[p * mn + i] - comp, z = sum + y;
    comp = fabsf(z) < __builtin_inff() ? (z - sum) - y : 0.f;
    sum = z;
  }
  c[(size_t)m * ldc + n] = sum * ((head_scales && head_dim > 0) ? head_scales[n / head_dim] : 1.0f);
}

template <typename TA, bool INT4, int MR, int WIN, int TW, int KS>
int launch_cm(hipStream_t s, const TA *a, const uint8_t *b, float *c, const float *sc, const float *hs, int M, int N,
              int K, int lda, int ldc, int hd, int kz = 1, float *part = nullptr) {
  const int nw = (K + WIN - 1) / WIN, nz = (nw + kz - 1) / kz, NI = (nz + KS - 1) / KS;
  const dim3 grid((unsigned)((gq_tiles(N) + TW - 1) / TW), (unsigned)((M + MR - 1) / MR), (unsigned)kz);
  hipLaunchKernelGGL((k_compat_mfma<INT4, TA, MR, WIN, TW, KS>), grid, dim3(64 * TW * KS), 0, s, a, b,
                     kz > 1 ? part : c, sc, kz > 1 ? nullptr : hs, M, N, K, lda, kz > 1 ? N : ldc, hd, NI);
  if (kz > 1)
    hipLaunchKernelGGL(k_cm_sum, dim3((unsigned)((N + 255) / 256), (unsigned)M), dim3(256), 0, s, part, hs, c, M, N,
                       ldc, hd, kz);
  return gq_last_launch();
}
// Whether the matrix-core form takes a shape: where the VALU kernels' time,
// which grows with M N K, passes the matrix cores' start-up (int4, VALU / matrix
// cores in us: 3 / 5 / 8 / 32 rows of 4096 x 4096 8.4 / 12.6 / 13.2 / 44.7 against 10.7 /
// 10.8 / 10.9 / 18.0, 8 / 32 rows of 1024 x 4096 7.0 / 13.0 against 10.5 / 16.8, 3 rows of
// 14336 x 4096 25.1 against 18.5; K <= 2048: 4 / 8 rows of 4096 x 2048 5.5 / 9.2 against 7.9 /
// 8.1, of 7000 x 1120 8.5 / 15.7 against 8.2 / 8.3; K <= 8192: 8 / 16 / 32 rows of 1024 x
// 6144 7.3 / 12.3 / 22.0 against 13.5 / 17.8 / 18.0, 4 / 5 rows of 4096 x 8192 17.5 / 23.8
// against 18.0; longer: 4 / 8 / 16 rows of 1024 x 14336 10.4 / 18.5 / 33.9 against 18.1 / 18.3 /
// 17.4.  The start-up grows with K: from 1024 x 6144 on a workgroup or two per CU
// walk several windows; past K = 8192 K goes over workgroups and it stops growing)
bool cm_takes(int M, int N, int K) {
  const double mnk = (double)M * N * K;
  const double from = K <= 2048 ? 40e6 : K <= 4096 && N >= 4096 ? 120e6 : K <= 8192 ? 160e6 : 120e6;
  return M >= 3 && mnk >= from;  // (two rows are one pass of the VALU kernels: 11.0 against 12.4 us, 14336 x 2048)
}
// Row tiles per workgroup and parts of K inside it (TW, KS) as the fp16 batch
// GEMV's plan; few row tiles on a long K, or more than 16 rows, take K in parts
// over workgroups as well (kz, sums in scratch): four row tiles then share the
// activations' limbs, whose making and reads otherwise outweigh the weights
// (int4, without / with: 16 rows of 4096 x 14336 38.3 / 26.9 us, 32 rows of 4096 x 4096
// 25.7 / 18.4, of 4096 x 14336 73.9 / 35.3; 8 rows of 4096 x 8192 18.3 / 19.1; 32 rows of
// 1024 x 2048, two parts, 8.5 / 16.3: the second launch is not worth two).
template <typename TA, bool INT4, int MR, int WIN>
int launch_cm_kz(hipStream_t s, const TA *a, const uint8_t *b, float *c, const float *sc, const float *hs, int M, int N,
                 int K, int lda, int ldc, int hd) {
  const size_t tiles = gq_tiles(N);
  const int nw = (K + WIN - 1) / WIN;
  const long wgs = (long)((tiles + 3) / 4) * ((M + MR - 1) / MR);
  const int kz = (int)(256 / wgs < nw / 8 ? 256 / wgs : nw / 8);
  if (tiles >= 800 || kz <= (K < 4096 ? 2 : 1) || (MR < 32 && K < 8192)) return GQ_ERR_UNSUPPORTED;
  GqScratch ws((size_t)kz * M * N * 4, s);
  if (!ws.ptr) return GQ_ERR_UNSUPPORTED;
  return launch_cm<TA, INT4, MR, WIN, 4, 4>(s, a, b, c, sc, hs, M, N, K, lda, ldc, hd, kz, (float *)ws.ptr);
}
template <typename TA, bool INT4, int MR, int WIN>
int launch_cm_plan(hipStream_t s, const TA *a, const uint8_t *b, float *c, const float *sc, const float *hs, int M,
                   int N, int K, int lda, int ldc, int hd) {
  const int r = launch_cm_kz<TA, INT4, MR, WIN>(s, a, b, c, sc, hs, M, N, K, lda, ldc, hd);
  if (r != GQ_ERR_UNSUPPORTED) return r;
  const size_t tiles = gq_tiles(N), wgs = (tiles + 3) / 4 * ((M + MR - 1) / MR);
  const int nw = (K + WIN - 1) / WIN;
#define GQ_CM(TW, KS) return launch_cm<TA, INT4, MR, WIN, TW, KS>(s, a, b, c, sc, hs, M, N, K, lda, ldc, hd)
  if constexpr (MR == 32) {
    // (fewer row tiles: 16 rows at a time on smaller workgroups)
    if (tiles < 400) return launch_cm_plan<TA, INT4, 16, WIN>(s, a, b, c, sc, hs, M, N, K, lda, ldc, hd);
  }
  // (a 16-wave workgroup fills a CU: two row tiles each past 512 would run in two
  // rounds; 9000 x 4096, two / four tiles: 4 / 8 / 16 rows int4 26.0 / 26.6 / 30.3 -> 18.0 / 19.0 /
  // 21.3 us, int8 38.5 / 38.7 / 33.5 -> 22.3 / 22.7 / 25.0)
  if (MR == 32 || tiles > 512) {
    // 8 waves, two workgroups to a CU, beyond one 16-wave workgroup each (int4: 8 rows
    // of 20000 x 2048 23.1 -> 19.2 us, of 28672 x 8192 63.5 -> 55.0; 32 rows 36.2 -> 29.5, 113 ->
    // 102) and, up to 8 rows, on a K whose walk is short (8 rows of 14336 x 1024 / 2048 / 4096 /
    // 6144 / 14336, 16 / 8 waves: int4 8.9 / 8.0, 12.9 / 11.9, 19.1 / 19.1, 27.0 / 27.6, 53 / 56; int8
    // 12.2 / 10.2, 16.6 / 14.3, 25.3 / 23.6, 35.0 / 33.7, 69.9 / 69.6)
    const bool short_walk = MR == 8 && K <= (INT4 ? 2048 : 6144);
    if (nw >= 2 && (wgs > 256 || short_walk)) GQ_CM(4, 2);
    if (nw >= 4) GQ_CM(4, 4);
    GQ_CM(4, 1);
  }
  if constexpr (MR < 32) {
    if (tiles >= 400) {
      // (up to 8 rows the 16 waves' budget of 128 registers spills: 6400 x 4096, 16 / 8
      // waves, int4 14.3 / 13.7, int8 20.8 / 16.0; 16 rows 16.3 / 17.7)
      if constexpr (MR == 16) {
        if (nw >= 8) GQ_CM(2, 8);
      }
      if (nw >= 4) GQ_CM(2, 4);
      GQ_CM(2, 1);
    }
    if (nw >= 8) GQ_CM(1, 8);
    if (nw >= 4) GQ_CM(1, 4);
    GQ_CM(1, 1);
  }
  return GQ_ERR_INVALID_ARGS;
#undef GQ_CM
}

template <typename TA, bool INT4>
int launch_compat(hipStream_t s, const TA *a, const uint8_t *b, float *c, const float *sc, const float *hs, int M,
                  int N, int K, int lda, int ldc, int gs, int srow, int hd) {
  const bool seg = K % 16 == 0 && (!sc || gs % 16 == 0) && lda % (sizeof(TA) == 4 ? 4 : 8) == 0 &&
                   (uintptr_t)a % 16 == 0 && (uintptr_t)b % 16 == 0;
  // (K % 32 and groups of 32: the two scale indexings agree and a group is a
  // row's own)
  if (seg && sc && gs == 32 && K % 32 == 0 && cm_takes(M, N, K)) {
    if (M <= 8) return launch_cm_plan<TA, INT4, 8, 256>(s, a, b, c, sc, hs, M, N, K, lda, ldc, hd);
    if (M <= 16) return launch_cm_plan<TA, INT4, 16, 128>(s, a, b, c, sc, hs, M, N, K, lda, ldc, hd);
    return launch_cm_plan<TA, INT4, 32, 128>(s, a, b, c, sc, hs, M, N, K, lda, ldc, hd);
  }
  // activations staged in LDS per 16-row workgroup (K <= 16384), else read
  // per wave (4096 x 4096 M = 1 / 8: 5.9 / 14.2 us against 7.5 / 20)
  if (seg && K <= 16384) {
    const int mb = (M >= 4 && K <= 4096) ? 4 : (M >= 2 && K <= 8192) ? 2 : 1;
    const size_t lds = (size_t)mb * K * 4;
    // INT4, one activation row, tall matrices: two rows per wave (twice the
    // weight bytes in flight per wave; 14336 x 4096: 14.3 -> 13.5 us) while
    // the grid keeps a workgroup per CU
    const bool rw2 = INT4 && mb == 1 && K <= 4096 && N >= 8192;
    dim3 grid((unsigned)((N + (rw2 ? 31 : 15)) / (rw2 ? 32 : 16)), (unsigned)((M + mb - 1) / mb));
    if (rw2) {
      hipLaunchKernelGGL((k_compat_gemv_lds<1, 4, TA, INT4, 2>), grid, dim3(1024), lds, s, a, b, c, sc, hs, M, N, K,
                         lda, ldc, gs, srow, hd);
      return gq_last_launch();
    }
#define GQ_LDS_L(MBV, NS)                                                                                       \
  hipLaunchKernelGGL((k_compat_gemv_lds<MBV, NS, TA, INT4>), grid, dim3(1024), lds, s, a, b, c, sc, hs, M, N, K, \
                     lda, ldc, gs, srow, hd)
    const int nseg = (K + 1023) / 1024;
    if (mb == 4) GQ_LDS_L(4, 4);
    else if (mb == 2) { if (nseg <= 4) GQ_LDS_L(2, 4); else GQ_LDS_L(2, 8); }
    else { if (nseg <= 4) GQ_LDS_L(1, 4); else if (nseg <= 8) GQ_LDS_L(1, 8); else GQ_LDS_L(1, 16); }
#undef GQ_LDS_L
    return gq_last_launch();
  }
  if (seg) {
    // MB activation rows per pass (the passes re-read the weights)
    const int mb = M >= 4 ? 4 : M >= 2 ? 2 : 1;
    dim3 grid((unsigned)((N + 15) / 16), (unsigned)((M + mb - 1) / mb));
    if (mb == 4)
      hipLaunchKernelGGL((k_compat_gemv_seg<4, 4, TA, INT4>), grid, dim3(256), 0, s, a, b, c, sc, hs, M, N, K, lda,
                         ldc, gs, srow, hd);
    else if (mb == 2)
      hipLaunchKernelGGL((k_compat_gemv_seg<2, 4, TA, INT4>), grid, dim3(256), 0, s, a, b, c, sc, hs, M, N, K, lda,
                         ldc, gs, srow, hd);
    else
      hipLaunchKernelGGL((k_compat_gemv_seg<1, 4, TA, INT4>), grid, dim3(256), 0, s, a, b, c, sc, hs, M, N, K, lda,
                         ldc, gs, srow, hd);
    return gq_last_launch();
  }
  dim3 grid((unsigned)((N + 3) / 4));
  for (int m = 0; m < M; m += 8)
    hipLaunchKernelGGL((k_compat_gemv<8, TA, INT4>), grid, dim3(256), 0, s, a, b, c, sc, hs, M, N, K, lda, ldc,
                       gs, srow, hd, m);
  return gq_last_launch();
}

// The reference's MFMA route (M > 32 without force_gemv: gemm_kernels.hip:
// 910-942, 742-760) computes on fp16 operands (A and w * s rounded to fp16);
// here the weights become Q8_0 / Q4_0 in T16 (d = fp16(s * h)) and go through
// gq_gemm.  Needs lda == K, ldc == N, K % 32 == 0 and
// gs % 32 == 0; the library's per-device workspace holds the converted
// weights (the launchers have no workspace argument).  GQ_ERR_UNSUPPORTED
// when a condition fails (the caller then runs the GEMV).
template <bool INT4>
int compat_gemm_route(hipStream_t s, const void *a, int a_dtype, const uint8_t *b, float *c, const float *sc,
                      const float *hs, int M, int N, int K, int lda, int ldc, int gs, int hd) {
  if (M <= 32 || lda != K || ldc != N || K % 32 || (sc && gs % 32)) return GQ_ERR_UNSUPPORTED;
  const int fmt = INT4 ? GQ_FMT_Q4_0 : GQ_FMT_Q8_0;
  const size_t packed = gq_align256(gq_packed_bytes(fmt, N, K));
  const size_t gws = gq_gemm_workspace_bytes(fmt, M, K);
  void *ws = nullptr;
  GQ_TRY(gq_default_workspace(packed + gws, &ws));
  uint8_t *wp = (uint8_t *)ws, *wa = wp + packed;
  GQ_TRY(gq_launch_rows_to_t16(INT4, b, sc, hs, N, K, gs, hd, wp, s));
  return gq_gemm(fmt, wp, a, a_dtype, c, GQ_DT_F32, M, N, K, wa, gws, s);
}

}  // namespace

extern "C" int gq_launch_gemm_mfma_int8_wt_fp32_acc32(void *stream, const float *a, const int8_t *b, float *c,
                                                       const float *scales, uint32_t M, uint32_t N, uint32_t K,
                                                       uint32_t lda, uint32_t ldb, uint32_t ldc,
                                                       uint32_t group_size) {
  (void)ldb;
  if (M == 0 || N == 0 || K == 0) return GQ_OK;
  GQ_CHECK(a && b && c, GQ_ERR_INVALID_ARGS);
  GQ_CHECK(!scales || group_size > 0, GQ_ERR_INVALID_ARGS);
  GQ_CHECK(M <= GQ_MAX_DIM && N <= GQ_MAX_DIM && K <= GQ_MAX_DIM, GQ_ERR_INVALID_ARGS);
  const int ld = (int)(lda ? lda : K), lc = (int)(ldc ? ldc : N);
  const int r = compat_gemm_route<false>((hipStream_t)stream, a, GQ_DT_F32, (const uint8_t *)b, c, scales, nullptr,
                                         (int)M, (int)N, (int)K, ld, lc, (int)group_size, 0);
  if (r != GQ_ERR_UNSUPPORTED) return r;
  // past the MFMA route's conditions the GEMV computes the MFMA route's scale
  // index for M > 32
  return launch_compat<float, false>((hipStream_t)stream, a, (const uint8_t *)b, c, scales, nullptr, (int)M, (int)N,
                                     (int)K, ld, lc, (int)group_size, M <= 32 ? 1 : 0, 0);
}

extern "C" int gq_launch_gemm_mfma_int4_wt_fp32_acc32(void *stream, const void *a, const int8_t *b, float *c,
                                                       const float *scales, const float *head_scales, uint32_t M,
                                                       uint32_t N, uint32_t K, uint32_t lda, uint32_t ldb,
                                                       uint32_t ldc, uint32_t group_size, uint32_t head_dim,
                                                       int is_fp16_a, int force_gemv) {
  (void)ldb;
  if (M == 0 || N == 0 || K == 0) return GQ_OK;
  GQ_CHECK(a && b && c, GQ_ERR_INVALID_ARGS);
  GQ_CHECK(!scales || group_size > 0, GQ_ERR_INVALID_ARGS);
  GQ_CHECK(M <= GQ_MAX_DIM && N <= GQ_MAX_DIM && K <= GQ_MAX_DIM, GQ_ERR_INVALID_ARGS);
  // the reference addresses row n at byte n*(K/2) (gemm_kernels.hip:781, 859)
  // while its loader packs the flat tensor (weight_loader.cpp:920-957): the
  // two agree only for even K
  GQ_CHECK(K % 2 == 0, GQ_ERR_UNSUPPORTED);
  hipStream_t s = (hipStream_t)stream;
  const int ld = (int)(lda ? lda : K), lc = (int)(ldc ? ldc : N);
  const int srow = (force_gemv || M <= 32) ? 1 : 0;  // the GEMV route's scale index
  if (!force_gemv) {  // the reference's MFMA route for M > 32
    const int r = compat_gemm_route<true>(s, a, is_fp16_a ? GQ_DT_F16 : GQ_DT_F32, (const uint8_t *)b, c, scales,
                                          head_scales, (int)M, (int)N, (int)K, ld, lc, (int)group_size,
                                          (int)head_dim);
    if (r != GQ_ERR_UNSUPPORTED) return r;
  }
  if (is_fp16_a)
    return launch_compat<_Float16, true>(s, (const _Float16 *)a, (const uint8_t *)b, c, scales, head_scales, (int)M,
                                         (int)N, (int)K, ld, lc, (int)group_size, srow, (int)head_dim);
  return launch_compat<float, true>(s, (const float *)a, (const uint8_t *)b, c, scales, head_scales, (int)M, (int)N,
                                    (int)K, ld, lc, (int)group_size, srow, (int)head_dim);
}
