// gq_quant.hip -- bit-exact GGUF dequantization, the T16 repack kernel and the
// activation preparation kernels used by the GEMV/GEMM paths.
//
// Dequantized values follow the reference semantics exactly:
//   Q4_K  src/inference/src/weight_loader.cpp:125-156 (products and the final
//         difference rounded separately -> contraction is disabled below)
//   Q8_0  weight_loader.cpp:703-712 + gemm_kernels.hip:612-616: (float)q * d
//   Q4_0  GGUF spec (no reference implementation): (float)(q - 8) * d
//   Q6_K  weight_loader.cpp:158-177: (d * (c - 32)) * scale
//   fp16  weight_loader.cpp:91-110 (NaN -> Inf)
#include "gq_internal.h"

#pragma clang fp contract(off)

namespace {

// ---------------------------------------------------------------------------
// Dequantization of raw GGUF blocks: one thread per 32 output elements.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256)
k_dequant_q4_0(const uint8_t *__restrict__ src, float *__restrict__ out, size_t nblk) {
  size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= nblk) return;
  const uint8_t *b = src + i * 18;
  float d = gq_h2f(gq_rd16(b));
  float y[32];
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    uint32_t q = b[2 + j];
    y[j] = (float)((int)(q & 15u) - 8) * d;
    y[j + 16] = (float)((int)(q >> 4) - 8) * d;
  }
  float4 *o = reinterpret_cast<float4 *>(out + i * 32);
#pragma unroll
  for (int v = 0; v < 8; ++v) o[v] = make_float4(y[4 * v], y[4 * v + 1], y[4 * v + 2], y[4 * v + 3]);
}

__global__ void __launch_bounds__(256)
k_dequant_q8_0(const uint8_t *__restrict__ src, float *__restrict__ out, size_t nblk) {
  size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= nblk) return;
  const uint8_t *b = src + i * 34;
  float d = gq_h2f(gq_rd16(b));
  float4 *o = reinterpret_cast<float4 *>(out + i * 32);
#pragma unroll
  for (int v = 0; v < 8; ++v) {
    float y0 = (float)(int8_t)b[2 + 4 * v] * d, y1 = (float)(int8_t)b[3 + 4 * v] * d;
    float y2 = (float)(int8_t)b[4 + 4 * v] * d, y3 = (float)(int8_t)b[5 + 4 * v] * d;
    o[v] = make_float4(y0, y1, y2, y3);
  }
}

// one thread per 32-element sub-block of a Q4_K super-block
__global__ void __launch_bounds__(256)
k_dequant_q4_k(const uint8_t *__restrict__ src, float *__restrict__ out, size_t nsub, int ggml) {
  size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= nsub) return;
  size_t sb = i >> 3;
  int j = (int)(i & 7);
  const uint8_t *b = src + sb * 144;
  float d = gq_h2f(gq_rd16(b)), dmin = gq_h2f(gq_rd16(b + 2));
  uint8_t sc[8], m[8];
  if (ggml) gq_q4k_ggml_codes(b + 4, sc, m);
  else gq_q4k_ref_codes(b + 4, sc, m);
  float scale = d * (float)sc[j];
  float minv = dmin * (float)m[j];
  float y[32];
#pragma unroll
  for (int e = 0; e < 32; ++e) {
    float p = scale * (float)gq_q4k_nib(ggml, b + 16, j, e);
    y[e] = p - minv;
  }
  float4 *o = reinterpret_cast<float4 *>(out + i * 32);
#pragma unroll
  for (int v = 0; v < 8; ++v) o[v] = make_float4(y[4 * v], y[4 * v + 1], y[4 * v + 2], y[4 * v + 3]);
}

// ---------------------------------------------------------------------------
// Dequantization straight from the T16 layout (proves the repack is lossless
// and gives the GEMM paths' weight values).  One thread per (row, 32-block).
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256)
k_dequant_t16(int fmt, const uint8_t *__restrict__ w, float *__restrict__ out, int N, int K) {
  size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  int nb = K / 32;
  if (i >= (size_t)N * nb) return;
  size_t n = i / nb, blk = i % nb;
  float y[32];
  const size_t C = gq_chunks(fmt, K);
  const uint8_t *scp = w + gq_sc_plane_offset(fmt, N, K);
  if (fmt == GQ_FMT_Q4_0) {
    float d = gq_h2f(gq_rd16(scp + gq_q4_0_d_off(n, blk, C)));
#pragma unroll
    for (int eh = 0; eh < 2; ++eh) {
      uint8_t c[16];
      gq_unpack_codes16(*reinterpret_cast<const uint64_t *>(w + gq_q4_0_grp_off(n, blk, eh, C)), c);
#pragma unroll
      for (int s = 0; s < 16; ++s) y[16 * eh + s] = (float)((int)c[s] - 8) * d;
    }
  } else if (fmt == GQ_FMT_Q8_0) {
    float d = gq_h2f(gq_rd16(scp + gq_q4_0_d_off(n, blk, C)));
#pragma unroll
    for (int eh = 0; eh < 2; ++eh) {
      const int8_t *q = reinterpret_cast<const int8_t *>(w + gq_q8_0_half_off(n, blk, eh, C));
#pragma unroll
      for (int s = 0; s < 16; ++s) y[16 * eh + s] = (float)q[s] * d;
    }
  } else if (fmt == GQ_FMT_Q6_K) {
    // (d * (c - 32)) * scale, as weight_loader.cpp:158-177 rounds it
    size_t s = blk >> 3;
    int j = (int)(blk & 7);
    const float d = gq_h2f(gq_rd16(scp + gq_q6k_d_off(n, s, C)));
    const int8_t *scl = reinterpret_cast<const int8_t *>(scp + gq_q6k_sc_off(n, s, C));
#pragma unroll
    for (int eh = 0; eh < 2; ++eh) {
      uint8_t c[16];
      gq_unpack_codes16(*reinterpret_cast<const uint64_t *>(w + gq_q6k_grp_off(n, s, j, eh, C)), c);
      const uint32_t hw = *reinterpret_cast<const uint32_t *>(w + gq_q6k_hi_off(n, s, j, eh, C));
      const float sc = (float)scl[2 * j + eh];
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const float p = d * (float)((int)(c[e] | (gq_q6k_hi_of(hw, e) << 4)) - 32);
        y[16 * eh + e] = p * sc;
      }
    }
  } else {
    size_t s = blk >> 3;
    int j = (int)(blk & 7);
    const uint32_t *meta = reinterpret_cast<const uint32_t *>(scp + gq_q4k_meta_off(n, s, C));
    uint32_t mv[4] = {meta[0], meta[1], meta[2], meta[3]};
    float d = gq_h2f(mv[0] & 0xFFFFu), dmin = gq_h2f(mv[0] >> 16);
    uint32_t scj, mj;
    gq_q4k_meta_codes(mv, j, &scj, &mj);
    float scale = d * (float)scj;
    float minv = dmin * (float)mj;
#pragma unroll
    for (int eh = 0; eh < 2; ++eh) {
      uint8_t c[16];
      gq_unpack_codes16(*reinterpret_cast<const uint64_t *>(w + gq_q4k_grp_off(n, s, j, eh, C)), c);
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        float p = scale * (float)c[e];
        y[16 * eh + e] = p - minv;
      }
    }
  }
  float4 *o = reinterpret_cast<float4 *>(out + n * (size_t)K + blk * 32);
#pragma unroll
  for (int v = 0; v < 8; ++v) o[v] = make_float4(y[4 * v], y[4 * v + 1], y[4 * v + 2], y[4 * v + 3]);
}

// ---------------------------------------------------------------------------
// Repack GGUF -> T16 of the rows [row0, row0 + rows) of an N-row tensor (row0 a
// multiple of 16; src points at row row0 of the GGUF data).
//
// Memory-bound: every byte is read and written once.  A workgroup takes one row
// tile and kSpan chunks of K: the 16 rows' segments (contiguous in the GGUF
// data, 544-840 bytes each) go to LDS in 16-byte loads, then each thread
// gathers 16-byte pieces of the T16 records from LDS and stores them in the
// records' order, so loads and stores are both coalesced and no code is touched
// byte by byte.  14336 x 4096 Q4_K: 110 us with one thread per block (144-byte
// strides, byte loads) -> 12.4 us; Q6_K 982 -> 16.8 us; 128256 x 4096 Q6_K 12.8 ms -> 150 us
// (5.7 TB/s read and written).  A row's last, partial span goes the same way
// up to its last whole 16 bytes (by byte pairs alone, 128256 x 256 took 23.7 us
// in Q4_0 and 35 in Q8_0, one thread per block 8.1 and 20.7).  Positions outside
// the tensor (rows past N, blocks past K) become zeros in LDS, so no memset is needed.
// ---------------------------------------------------------------------------
template <int FMT>
struct RpFmt;  // per row and chunk: GGUF bytes; 16-byte pieces of the code record and of the scale record
template <>
struct RpFmt<GQ_FMT_Q4_0> {
  static constexpr int kBytes = 72, kSpan = 8, kQs = 64, kSc = 8;
};
template <>
struct RpFmt<GQ_FMT_Q8_0> {
  static constexpr int kBytes = 136, kSpan = 4, kQs = 128, kSc = 8;
};
template <>
struct RpFmt<GQ_FMT_Q4_K> {
  static constexpr int kBytes = 144, kSpan = 4, kQs = 128, kSc = 16;
};
template <>
struct RpFmt<GQ_FMT_Q6_K> {
  static constexpr int kBytes = 210, kSpan = 4, kQs = 192, kSc = 18;
};

struct __attribute__((packed)) RpLoad16 {  // a GGUF row starts at any byte
  gq_u4 v;
};

// 4 dwords at LDS byte p + off (off a multiple of 2, p of 4)
GQ_DEV gq_u4 rp_ld16(const uint8_t *p, int off) {
  const uint32_t *q = reinterpret_cast<const uint32_t *>(p + (off & ~3));
  const uint32_t d[5] = {q[0], q[1], q[2], q[3], q[4]};
  const uint32_t sh = 8u * (uint32_t)(off & 2);
  gq_u4 o;
#pragma unroll
  for (int i = 0; i < 4; ++i) o[i] = __builtin_amdgcn_alignbit(d[i + 1], d[i], sh);
  return o;
}
GQ_DEV gq_u2 rp_ld8(const uint8_t *p, int off) {
  const uint32_t *q = reinterpret_cast<const uint32_t *>(p + (off & ~3));
  const uint32_t sh = 8u * (uint32_t)(off & 2);
  return gq_u2{__builtin_amdgcn_alignbit(q[1], q[0], sh), __builtin_amdgcn_alignbit(q[2], q[1], sh)};
}
GQ_DEV uint32_t rp_ld2(const uint8_t *p, int off) { return *reinterpret_cast<const uint16_t *>(p + off); }

// 16 codes, one per byte (nibble `hi` of the 16 bytes v) -> the code group
GQ_DEV gq_u2 rp_group_bytes(gq_u4 v, int hi) {
  const uint32_t m = 0x0F0F0F0Fu, sh = 4u * (uint32_t)hi;
  return gq_u2{((v[0] >> sh) & m) | (((v[1] >> sh) & m) << 4), ((v[2] >> sh) & m) | (((v[3] >> sh) & m) << 4)};
}
// four nibbles (16 bits) -> the low nibbles of four bytes
GQ_DEV uint32_t rp_spread(uint32_t x) {
  x = (x | (x << 8)) & 0x00FF00FFu;
  return (x | (x << 4)) & 0x0F0F0F0Fu;
}
// 16 codes in element order, two per byte -> the code group
GQ_DEV gq_u2 rp_group_nibs(gq_u2 v) {
  return gq_u2{rp_spread(v[0] & 0xFFFFu) | (rp_spread(v[0] >> 16) << 4),
               rp_spread(v[1] & 0xFFFFu) | (rp_spread(v[1] >> 16) << 4)};
}
// 16 two-bit fields in element order, field 4 q + b at bits 8 q + 2 b -> at bits
// 8 b + 2 q (a 4 x 4 transpose by two exchanges)
GQ_DEV uint32_t rp_hi_transpose(uint32_t x) {
  uint32_t t = ((x >> 6) ^ x) & 0x00CC00CCu;
  x ^= t ^ (t << 6);
  t = ((x >> 12) ^ x) & 0x0000F0F0u;
  return x ^ t ^ (t << 12);
}

// code group of 32-block j, half eh of the chunk at LDS bytes p + o
template <int FMT>
GQ_DEV gq_u2 rp_group(const uint8_t *p, int o, int j, int eh, int ggml) {
  if constexpr (FMT == GQ_FMT_Q4_0) return rp_group_bytes(rp_ld16(p, o + 18 * j + 2), eh);
  if constexpr (FMT == GQ_FMT_Q4_K) {
    if (ggml) return rp_group_bytes(rp_ld16(p, o + 16 + 32 * (j >> 1) + 16 * eh), j & 1);
    return rp_group_nibs(rp_ld8(p, o + 16 + 16 * j + 8 * eh));
  }
  if (ggml) return rp_group_bytes(rp_ld16(p, o + 64 * (j >> 2) + 16 * eh + 32 * (j & 1)), (j >> 1) & 1);
  return rp_group_nibs(rp_ld8(p, o + 16 * j + 8 * eh));
}
// Q6_K: the high fields of 32-block j, half eh as the T16 word
GQ_DEV uint32_t rp_hi(const uint8_t *p, int o, int j, int eh, int ggml) {
  if (!ggml) {
    const int at = o + 128 + 8 * j + 4 * eh;
    return rp_hi_transpose(rp_ld2(p, at) | (rp_ld2(p, at + 2) << 16));
  }
  const gq_u4 v = rp_ld16(p, o + 128 + 32 * (j >> 2) + 16 * eh);
  uint32_t h = 0;
#pragma unroll
  for (int q = 0; q < 4; ++q) h |= ((v[q] >> (2 * (j & 3))) & 0x03030303u) << (2 * q);
  return h;
}

template <int FMT, int kSpan = RpFmt<FMT>::kSpan, int NT = 256>
__global__ void __launch_bounds__(NT)
k_repack(const uint8_t *__restrict__ src, uint8_t *__restrict__ dst, size_t sc_off, int N, size_t row_bytes, int C,
         int row0, int ggml) {
  using F = RpFmt<FMT>;
  constexpr int SEG = F::kBytes * kSpan;        // a multiple of 8
  constexpr int UPR = (SEG + 15) / 16;             // 16-byte loads per row
  constexpr int PITCH = (UPR * 4 + 2) * 4 + 4;     // an odd count of dwords: the 16 rows on different banks
  static_assert((PITCH / 4) % 2 == 1 && PITCH >= UPR * 16 + 4, "LDS pitch");
  constexpr int LD = (16 * UPR + NT - 1) / NT;
  __shared__ __attribute__((aligned(16))) uint8_t seg[16 * PITCH];
  const int nsp = (C + kSpan - 1) / kSpan;
  const int t = (int)(blockIdx.x / (unsigned)nsp), c0 = (int)(blockIdx.x % (unsigned)nsp) * kSpan;  // tile of the slice
  const int tid = threadIdx.x;
  const int nrows = min(16, N - (row0 + 16 * t));  // rows inside the tensor (>= 1)
  const size_t sb = (size_t)c0 * F::kBytes;
  const size_t left = row_bytes - sb;
  const uint8_t *base = src + (size_t)(16 * t) * row_bytes + sb;
  if (left >= (size_t)SEG) {
    // whole segments: unconditional loads (the last one of a row moved back to
    // end with it), rows past N zeroed after
    gq_u4 v[LD];
#pragma unroll
    for (int q = 0; q < LD; ++q) {
      const int i = tid + NT * q, row = min(i / UPR, nrows - 1), o = min(16 * (i % UPR), SEG - 16);
      v[q] = reinterpret_cast<const RpLoad16 *>(base + (size_t)row * row_bytes + o)->v;
    }
#pragma unroll
    for (int q = 0; q < LD; ++q) {
      const int i = tid + NT * q, row = i / UPR, o = min(16 * (i % UPR), SEG - 16);
      if (row < 16) {
        uint32_t *d = reinterpret_cast<uint32_t *>(seg + row * PITCH + o);
#pragma unroll
        for (int e = 0; e < 4; ++e) d[e] = row < nrows ? v[q][e] : 0u;
      }
    }
  } else {
    // the row's end (a short row's only segment): whole pieces of 16, then byte
    // pairs, zeros past the row up to the last chunk's end
    const int full = (int)left >> 4, end = min(kSpan, C - c0) * F::kBytes;
    gq_u4 v[LD];
#pragma unroll
    for (int q = 0; q < LD; ++q) {
      const int i = tid + NT * q, row = min(i / UPR, nrows - 1), u = min(i % UPR, full - 1);
      if (full > 0) v[q] = reinterpret_cast<const RpLoad16 *>(base + (size_t)row * row_bytes + 16 * u)->v;
    }
#pragma unroll
    for (int q = 0; q < LD; ++q) {
      const int i = tid + NT * q, row = i / UPR, u = i % UPR;
      if (row < 16 && u < full) {
        uint32_t *d = reinterpret_cast<uint32_t *>(seg + row * PITCH + 16 * u);
#pragma unroll
        for (int e = 0; e < 4; ++e) d[e] = row < nrows ? v[q][e] : 0u;
      }
    }
    for (int i = tid >> 4; i < (end >> 1) - 8 * full; i += NT / 16) {
      const int row = tid & 15, o = 16 * full + 2 * i;
      uint32_t x = 0;
      if (row < nrows && (size_t)o + 2 <= left) {
        const uint8_t *p = base + (size_t)row * row_bytes + o;
        x = (uint32_t)p[0] | ((uint32_t)p[1] << 8);
      }
      *reinterpret_cast<uint16_t *>(seg + row * PITCH + o) = (uint16_t)x;
    }
  }
  __syncthreads();
  const int nc = min(kSpan, C - c0);
  const size_t tc = (size_t)(row0 / 16 + t) * (size_t)C + (size_t)c0;
  gq_u4 *qs = reinterpret_cast<gq_u4 *>(dst + tc * (16 * F::kQs));
  for (int i = tid; i < nc * F::kQs; i += NT) {
    const int c = i / F::kQs, pc = i % F::kQs, l = pc & 63, part = pc >> 6;
    const int r = l & 15, g = l >> 4, eh = g & 1, jh = g >> 1;
    const uint8_t *p = seg + r * PITCH;
    const int o = c * F::kBytes;
    gq_u4 v;
    if constexpr (FMT == GQ_FMT_Q8_0) {
      v = rp_ld16(p, o + 34 * (2 * part + jh) + 2 + 16 * eh);
    } else {
      if (FMT == GQ_FMT_Q6_K && part == 2) {
#pragma unroll
        for (int m = 0; m < 4; ++m) v[m] = rp_hi(p, o, 2 * m + jh, eh, ggml);
      } else {
        const gq_u2 a = rp_group<FMT>(p, o, 4 * part + jh, eh, ggml);
        const gq_u2 b = rp_group<FMT>(p, o, 4 * part + 2 + jh, eh, ggml);
        v = gq_u4{a[0], a[1], b[0], b[1]};
      }
    }
    qs[i] = v;
  }
  gq_u4 *sc = reinterpret_cast<gq_u4 *>(dst + sc_off + tc * (16 * F::kSc));
  for (int i = tid; i < nc * F::kSc; i += NT) {
    const int c = i / F::kSc, pc = i % F::kSc;
    const int o = c * F::kBytes;
    gq_u4 v;
    if constexpr (FMT == GQ_FMT_Q4_0 || FMT == GQ_FMT_Q8_0) {
      // two rows' block scales, in the order d0 d2 d1 d3
      constexpr int BB = F::kBytes / 4;
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const uint8_t *p = seg + (2 * pc + e) * PITCH;
        v[2 * e] = rp_ld2(p, o) | (rp_ld2(p, o + 2 * BB) << 16);
        v[2 * e + 1] = rp_ld2(p, o + BB) | (rp_ld2(p, o + 3 * BB) << 16);
      }
    } else if constexpr (FMT == GQ_FMT_Q4_K) {
      const uint8_t *p = seg + pc * PITCH + o;
      uint8_t s[12], scc[8], m[8];
#pragma unroll
      for (int e = 0; e < 12; ++e) s[e] = p[4 + e];
      if (ggml) gq_q4k_ggml_codes(s, scc, m);
      else gq_q4k_ref_codes(s, scc, m);
      uint32_t w1 = 0, w2 = 0, w3 = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t m0 = m[2 * e], m1 = m[2 * e + 1];
        w1 |= ((uint32_t)scc[2 * e] | ((m0 & 3u) << 6)) << (8 * e);
        w2 |= ((uint32_t)scc[2 * e + 1] | ((m1 & 3u) << 6)) << (8 * e);
        w3 |= ((m0 >> 2) | ((m1 >> 2) << 4)) << (8 * e);
      }
      v = gq_u4{*reinterpret_cast<const uint32_t *>(p), w1, w2, w3};
    } else if (pc < 16) {
      v = rp_ld16(seg + pc * PITCH, o + 192);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint8_t *p = seg + (8 * (pc - 16) + 2 * e) * PITCH;
        v[e] = rp_ld2(p, o + 208) | (rp_ld2(p + PITCH, o + 208) << 16);
      }
    }
    sc[i] = v;
  }
}

// Reference INT8 / INT4 rows -> T16 Q8_0 / Q4_0 for the launchers' MFMA route:
// INT8 codes as they are, INT4 codes q (two's complement, even k in the low
// nibble) as q + 8; d = fp16(s * h), the group's scale times the row's head factor.
// The same work split as k_repack (a row tile and 512 bytes of each row), so the
// codes pass through memory once each way: 4096 x 4096 INT8 8.8 us against 8 + 6.8 (and their gap) for
// blocks first and their repack.  K % 32 == 0, gs % 32 == 0 (host-checked).
template <bool INT4>
__global__ void __launch_bounds__(256)
k_rows_to_t16(const uint8_t *__restrict__ b, const float *__restrict__ scales, const float *__restrict__ hs,
              uint8_t *__restrict__ dst, size_t sc_off, int N, int K, int C, int gs, int head_dim) {
  constexpr int CB = INT4 ? 64 : 128, SPAN = 512 / CB;  // bytes of a row per chunk; chunks
  constexpr int PITCH = 512 + 4;                        // (an odd count of dwords)
  constexpr int QS = INT4 ? 64 : 128;                   // 16-byte pieces per chunk
  __shared__ __attribute__((aligned(16))) uint8_t seg[16 * PITCH];
  const int nsp = (C + SPAN - 1) / SPAN;
  const int t = (int)(blockIdx.x / (unsigned)nsp), c0 = (int)(blockIdx.x % (unsigned)nsp) * SPAN;
  const int tid = threadIdx.x, nb = K / 32;
  const size_t row_bytes = (size_t)K * CB / 128;
  const int left = (int)(row_bytes - (size_t)c0 * CB);  // a multiple of 16
  gq_u4 v[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int i = tid + 256 * q, row = min(16 * t + (i >> 5), N - 1), o = 16 * (i & 31);
    v[q] = reinterpret_cast<const RpLoad16 *>(b + (size_t)row * row_bytes + (size_t)c0 * CB + (o < left ? o : 0))->v;
  }
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int i = tid + 256 * q, o = 16 * (i & 31);
    const bool in = 16 * t + (i >> 5) < N && o < left;
    uint32_t *d = reinterpret_cast<uint32_t *>(seg + (i >> 5) * PITCH + o);
#pragma unroll
    for (int e = 0; e < 4; ++e) d[e] = in ? (INT4 ? v[q][e] ^ 0x88888888u : v[q][e]) : 0u;
  }
  __syncthreads();
  const int nc = min(SPAN, C - c0);
  const size_t tc = (size_t)t * (size_t)C + (size_t)c0;
  gq_u4 *qs = reinterpret_cast<gq_u4 *>(dst + tc * (16 * QS));
  for (int i = tid; i < nc * QS; i += 256) {
    const int c = i / QS, pc = i % QS, l = pc & 63, part = pc >> 6;
    const int r = l & 15, g = l >> 4, eh = g & 1, jh = g >> 1;
    const uint8_t *p = seg + r * PITCH + c * CB;
    if constexpr (INT4) {
      const uint32_t *w0 = reinterpret_cast<const uint32_t *>(p + 16 * jh + 8 * eh);
      const uint32_t *w1 = reinterpret_cast<const uint32_t *>(p + 16 * (2 + jh) + 8 * eh);
      const gq_u2 a = rp_group_nibs(gq_u2{w0[0], w0[1]}), e = rp_group_nibs(gq_u2{w1[0], w1[1]});
      qs[i] = gq_u4{a[0], a[1], e[0], e[1]};
    } else {
      const uint32_t *w = reinterpret_cast<const uint32_t *>(p + 32 * (2 * part + jh) + 16 * eh);
      qs[i] = gq_u4{w[0], w[1], w[2], w[3]};
    }
  }
  // one row's four block scales of a chunk per thread, in the order d0 d2 d1 d3
  gq_u2 *sc = reinterpret_cast<gq_u2 *>(dst + sc_off + tc * 128);
  for (int i = tid; i < nc * 16; i += 256) {
    const int c = i >> 4, n = 16 * t + (i & 15), b0 = 4 * (c0 + c);
    uint32_t d[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const bool in = n < N && b0 + j < nb;
      float s = 1.0f;
      if (in) {
        if (scales) s = scales[((size_t)n * K + 32 * (size_t)(b0 + j)) / (size_t)gs];
        if (hs && head_dim > 0) s *= hs[n / head_dim];
      }
      d[j] = in ? __builtin_bit_cast(uint16_t, (_Float16)s) : 0u;
    }
    sc[i] = gq_u2{d[0] | (d[2] << 16), d[1] | (d[3] << 16)};
  }
}

template <int FMT>
void launch_repack(const uint8_t *src, uint8_t *dst, size_t N, size_t K, size_t row0, size_t tiles, int ggml,
                   hipStream_t s) {
  const size_t C = gq_chunks(FMT, K), nsp = (C + RpFmt<FMT>::kSpan - 1) / RpFmt<FMT>::kSpan;
  // one or two chunks a row leave a workgroup little: one wave takes them
  // (128256 x 256, Q4_0 10.4 -> 6.9 us, Q8_0 13.4 -> 12.8)
  if constexpr (FMT == GQ_FMT_Q4_0 || FMT == GQ_FMT_Q8_0) {
    if (C <= 2) {
      hipLaunchKernelGGL((k_repack<FMT, 2, 64>), dim3((unsigned)tiles), dim3(64), 0, s, src, dst,
                         gq_sc_plane_offset(FMT, N, K), (int)N, gq_layout_gguf_bytes(FMT, 1, K), (int)C, (int)row0, ggml);
      return;
    }
  }
  hipLaunchKernelGGL(k_repack<FMT>, dim3((unsigned)(tiles * nsp)), dim3(256), 0, s, src, dst,
                     gq_sc_plane_offset(FMT, N, K), (int)N, gq_layout_gguf_bytes(FMT, 1, K), (int)C, (int)row0, ggml);
}

// ---------------------------------------------------------------------------
// Activation preparation for the GEMV with batch > 4.  x f32 [B][K] ->
//   limbs int8 [B][2][Kp]: x ~ s * (a + b / 254) per 32-block, s = amax / 127
//   zero  int8 [Kp]
//   scl   float4 [B][Kp/32]: (s, S, s / 254, 0), S = sum of the represented block
// Elements k >= K are zeros.  One thread per 32-block.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256)
k_prep_x(const float *__restrict__ x, int8_t *__restrict__ xl, float *__restrict__ scl, int B, int K, int Kp) {
  const int nblk = Kp / 32;
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= B * nblk) return;
  const int b = i / nblk, j = i % nblk;
  const float *xr = x + (size_t)b * K + 32 * j;
  float v[32];
  if (32 * j + 32 <= K) {
    const float4 *p = reinterpret_cast<const float4 *>(xr);
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const float4 t = p[q];
      v[4 * q] = t.x; v[4 * q + 1] = t.y; v[4 * q + 2] = t.z; v[4 * q + 3] = t.w;
    }
  } else {
#pragma unroll
    for (int e = 0; e < 32; ++e) v[e] = 0.0f;
  }
  float amax = 0.f, s = 0.f;
#pragma unroll
  for (int e = 0; e < 32; ++e) amax = fmaxf(amax, fabsf(v[e]));
  const float inv = amax > 0.f ? 127.0f / amax : 0.f;
  const float sx = amax * (1.0f / 127.0f);
  uint32_t la[8], lb[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    uint32_t wa = 0, wb = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float t = v[4 * q + e] * inv;
      const float a = rintf(t);
      const float bb = rintf((t - a) * 254.0f);
      s += a * 254.0f + bb;  // exact integer
      wa |= ((uint32_t)(int)a & 0xFFu) << (8 * e);
      wb |= ((uint32_t)(int)bb & 0xFFu) << (8 * e);
    }
    la[q] = wa;
    lb[q] = wb;
  }
  gq_u4 *pa = reinterpret_cast<gq_u4 *>(xl + (size_t)(2 * b) * Kp + 32 * j);
  gq_u4 *pb = reinterpret_cast<gq_u4 *>(xl + (size_t)(2 * b + 1) * Kp + 32 * j);
  pa[0] = gq_u4{la[0], la[1], la[2], la[3]};
  pa[1] = gq_u4{la[4], la[5], la[6], la[7]};
  pb[0] = gq_u4{lb[0], lb[1], lb[2], lb[3]};
  pb[1] = gq_u4{lb[4], lb[5], lb[6], lb[7]};
  if (b == 0) {
    gq_u4 *pz = reinterpret_cast<gq_u4 *>(xl + (size_t)2 * B * Kp + 32 * j);
    pz[0] = gq_u4{0u, 0u, 0u, 0u};
    pz[1] = gq_u4{0u, 0u, 0u, 0u};
  }
  s *= sx * (1.0f / 254.0f);  // block sum of the represented values
  *reinterpret_cast<gq_f4 *>(scl + 4 * ((size_t)b * nblk + j)) = gq_f4{sx, s, sx * (1.0f / 254.0f), 0.f};
}

// Per-32 int8 activation quantization (Q8_0 int8-MFMA path): the reference's
// INT8 requant rule applied to activations (weight_loader.cpp:780-802):
// d = amax/127, inv = d > 1e-9 ? 1/d : 0, q = round(a * inv), half away.
// Four lanes per block, 8 elements each in 16-byte loads (one thread per block
// read 128 bytes at that stride: 512 x 4096 fp32 9.5 -> 4.6 us).
template <typename T>
struct __attribute__((packed)) QaLoad8 {  // (A starts at any element)
  T v[8];
};
template <int DT>
__global__ void __launch_bounds__(256)
k_quantize_act_q8(const void *__restrict__ a, int8_t *__restrict__ q, float *__restrict__ dq, size_t n8) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;  // run of 8 (rows are whole blocks)
  const size_t at = i < n8 ? i : n8 - 1;
  float v[8];
  if constexpr (DT == GQ_DT_F32) {
    const auto t = reinterpret_cast<const QaLoad8<float> *>(a)[at];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = t.v[e];
  } else {
    const auto t = reinterpret_cast<const QaLoad8<uint16_t> *>(a)[at];
#pragma unroll
    for (int e = 0; e < 8; ++e)
      v[e] = DT == GQ_DT_BF16 ? __uint_as_float((uint32_t)t.v[e] << 16)
                              : (float)__builtin_bit_cast(_Float16, t.v[e]);
  }
  float mx = 0.0f;
#pragma unroll
  for (int e = 0; e < 8; ++e) mx = fmaxf(mx, fabsf(v[e]));
  mx = fmaxf(mx, __shfl_xor(mx, 1, 64));
  mx = fmaxf(mx, __shfl_xor(mx, 2, 64));
  const float d = mx / 127.0f;
  const float inv = d > 1e-9f ? 1.0f / d : 0.0f;
  uint32_t words[2] = {0, 0};
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int qi = (int)roundf(v[e] * inv);
    words[e >> 2] |= ((uint32_t)qi & 0xFFu) << (8 * (e & 3));
  }
  if (i >= n8) return;
  reinterpret_cast<gq_u2 *>(q)[i] = gq_u2{words[0], words[1]};
  if ((i & 3) == 0) dq[i >> 2] = d;
}

}  // namespace

static unsigned blocks_for(size_t n) { return (unsigned)((n + 255) / 256); }

extern "C" int gq_dequant_gguf(int fmt, const void *blocks, size_t n_blocks, float *out, void *stream) {
  GQ_CHECK(gq_fmt_valid(fmt) || fmt == GQ_FMT_F16, GQ_ERR_UNSUPPORTED);
  GQ_CHECK(blocks && out, GQ_ERR_INVALID_ARGS);
  if (n_blocks == 0) return GQ_OK;
  hipStream_t s = (hipStream_t)stream;
  if (fmt == GQ_FMT_F16) return gq_launch_f16_to_f32(blocks, n_blocks, out, s);
  if (gq_fmt_is_q6k(fmt)) return gq_launch_dequant_q6_k(blocks, n_blocks, out, fmt == GQ_FMT_Q6_K_GGML, s);
  const uint8_t *src = (const uint8_t *)blocks;
  if (fmt == GQ_FMT_Q4_0)
    hipLaunchKernelGGL(k_dequant_q4_0, dim3(blocks_for(n_blocks)), dim3(256), 0, s, src, out, n_blocks);
  else if (fmt == GQ_FMT_Q8_0)
    hipLaunchKernelGGL(k_dequant_q8_0, dim3(blocks_for(n_blocks)), dim3(256), 0, s, src, out, n_blocks);
  else
    hipLaunchKernelGGL(k_dequant_q4_k, dim3(blocks_for(n_blocks * 8)), dim3(256), 0, s, src, out,
                       n_blocks * 8, (int)(fmt == GQ_FMT_Q4_K_GGML));
  return gq_last_launch();
}

extern "C" int gq_dequant_packed(int fmt, const void *packed, size_t N, size_t K, float *out, void *stream) {
  GQ_TRY(gq_check_shape(fmt, N, K));
  GQ_CHECK(packed && out, GQ_ERR_INVALID_ARGS);
  if (N == 0 || K == 0) return GQ_OK;
  int f = gq_fmt_is_q4k(fmt) ? GQ_FMT_Q4_K : gq_fmt_is_q6k(fmt) ? GQ_FMT_Q6_K : fmt;
  hipLaunchKernelGGL(k_dequant_t16, dim3(blocks_for(N * (K / 32))), dim3(256), 0, (hipStream_t)stream, f,
                     (const uint8_t *)packed, out, (int)N, (int)K);
  return gq_last_launch();
}

extern "C" int gq_repack_rows(int fmt, const void *gguf_rows, size_t N, size_t K, size_t row0, size_t rows,
                              void *packed, void *stream) {
  GQ_TRY(gq_check_shape(fmt, N, K));
  GQ_CHECK(gguf_rows && packed, GQ_ERR_INVALID_ARGS);
  GQ_CHECK(row0 % 16 == 0 && row0 <= N && rows <= N - row0, GQ_ERR_INVALID_ARGS);
  GQ_CHECK(row0 + rows == N || rows % 16 == 0, GQ_ERR_INVALID_ARGS);  // whole tiles, or the tensor's end
  if (rows == 0 || K == 0) return GQ_OK;
  hipStream_t s = (hipStream_t)stream;
  // whole tiles: the padding rows of the last one are zeroed
  const size_t tiles = gq_tiles(rows);
  const uint8_t *src = (const uint8_t *)gguf_rows;
  uint8_t *dst = (uint8_t *)packed;
  if (fmt == GQ_FMT_Q4_0) launch_repack<GQ_FMT_Q4_0>(src, dst, N, K, row0, tiles, 0, s);
  else if (fmt == GQ_FMT_Q8_0) launch_repack<GQ_FMT_Q8_0>(src, dst, N, K, row0, tiles, 0, s);
  else if (gq_fmt_is_q6k(fmt)) launch_repack<GQ_FMT_Q6_K>(src, dst, N, K, row0, tiles, fmt == GQ_FMT_Q6_K_GGML, s);
  else launch_repack<GQ_FMT_Q4_K>(src, dst, N, K, row0, tiles, fmt == GQ_FMT_Q4_K_GGML, s);
  return gq_last_launch();
}

int gq_launch_rows_to_t16(bool int4, const void *b, const float *scales, const float *head_scales, int N, int K, int gs,
                          int head_dim, void *packed, hipStream_t s) {
  const int fmt = int4 ? GQ_FMT_Q4_0 : GQ_FMT_Q8_0, C = (int)gq_chunks(fmt, K), span = int4 ? 8 : 4;
  const dim3 grid((unsigned)(gq_tiles(N) * ((C + span - 1) / span)));
  const size_t sc_off = gq_sc_plane_offset(fmt, N, K);
  if (int4)
    hipLaunchKernelGGL(k_rows_to_t16<true>, grid, dim3(256), 0, s, (const uint8_t *)b, scales, head_scales,
                       (uint8_t *)packed, sc_off, N, K, C, gs, head_dim);
  else
    hipLaunchKernelGGL(k_rows_to_t16<false>, grid, dim3(256), 0, s, (const uint8_t *)b, scales, head_scales,
                       (uint8_t *)packed, sc_off, N, K, C, gs, head_dim);
  return gq_last_launch();
}

extern "C" int gq_repack(int fmt, const void *gguf, size_t N, size_t K, void *packed, void *stream) {
  return gq_repack_rows(fmt, gguf, N, K, 0, N, packed, stream);
}

int gq_launch_prep_x(int fmt, const float *x, void *ws, int B, int K, hipStream_t s) {
  const int Kp = (int)gq_kpad(fmt, K);
  int8_t *xl = (int8_t *)ws;
  float *scl = (float *)((uint8_t *)ws + gq_xl_bytes(fmt, K, B));
  const int n = B * (Kp / 32);
  hipLaunchKernelGGL(k_prep_x, dim3(blocks_for(n)), dim3(256), 0, s, x, xl, scl, B, K, Kp);
  return gq_last_launch();
}

namespace {
__global__ void __launch_bounds__(256) k_fill_zero(float *p, size_t n) {
  size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) p[i] = 0.0f;
}
}  // namespace

int gq_fill_zero(float *p, size_t n, hipStream_t s) {
  if (n == 0) return GQ_OK;
  hipLaunchKernelGGL(k_fill_zero, dim3(blocks_for(n)), dim3(256), 0, s, p, n);
  return gq_last_launch();
}


extern "C" int gq_quantize_act_q8(const void *a, int a_dtype, size_t M, size_t K, int8_t *q, float *d,
                                  void *stream) {
  GQ_CHECK(a && q && d, GQ_ERR_INVALID_ARGS);
  GQ_CHECK(a_dtype == GQ_DT_F32 || a_dtype == GQ_DT_F16 || a_dtype == GQ_DT_BF16, GQ_ERR_UNSUPPORTED);
  GQ_CHECK(K % 32 == 0 && K <= GQ_MAX_DIM && M <= GQ_MAX_DIM, GQ_ERR_INVALID_ARGS);
  if (M == 0 || K == 0) return GQ_OK;
  const size_t n8 = M * (K / 8);
  const dim3 grid(blocks_for(n8));
  if (a_dtype == GQ_DT_F32)
    hipLaunchKernelGGL(k_quantize_act_q8<GQ_DT_F32>, grid, dim3(256), 0, (hipStream_t)stream, a, q, d, n8);
  else if (a_dtype == GQ_DT_F16)
    hipLaunchKernelGGL(k_quantize_act_q8<GQ_DT_F16>, grid, dim3(256), 0, (hipStream_t)stream, a, q, d, n8);
  else
    hipLaunchKernelGGL(k_quantize_act_q8<GQ_DT_BF16>, grid, dim3(256), 0, (hipStream_t)stream, a, q, d, n8);
  return gq_last_launch();
}
