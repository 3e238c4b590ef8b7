// gq_internal.h -- shared declarations of the libgq implementation files.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "../../include/gq.h"
#include "gq_device.h"
#include "gq_layout.h"
#include "gq_repack_impl.h"

#define GQ_CHECK(cond, code) \
  do {                       \
    if (!(cond)) return (code); \
  } while (0)
#define GQ_TRY(expr)          \
  do {                        \
    int _st = (expr);         \
    if (_st != GQ_OK) return _st; \
  } while (0)

// Records the HIP error (if any) of the last launch and maps it to a status.
int gq_last_launch(void);
int gq_hip_status(hipError_t e);

// Validates (fmt, N, K): known format, K a multiple of the block size, sizes
// within GQ_MAX_DIM.
static inline int gq_check_shape(int fmt, size_t N, size_t K) {
  if (!gq_fmt_valid(fmt)) return GQ_ERR_UNSUPPORTED;
  if (N > GQ_MAX_DIM || K > GQ_MAX_DIM) return GQ_ERR_INVALID_ARGS;
  if (K % gq_block_elems(fmt)) return GQ_ERR_INVALID_ARGS;
  return GQ_OK;
}

static inline size_t gq_align256(size_t v) { return (v + 255) & ~(size_t)255; }
// padded K of the T16 layout
static inline size_t gq_kpad(int fmt, size_t K) { return gq_chunks(fmt, K) * gq_chunk_k(fmt); }
// padded K of the tiled GEMM on fp16 weights (four 64-k steps: its K groups)
static inline size_t gq_f16w_kpad(size_t K) { return (K + 255) & ~(size_t)255; }
// GEMV workspace (batch > 4): int8 limbs [B][2][Kp] then a zero region of Kp
// bytes, then per (batch row, 32-block) float4 (s, S, s / 254, 0).
static inline size_t gq_xl_bytes(int fmt, size_t K, int B) {
  return gq_align256(((size_t)2 * B + 1) * gq_kpad(fmt, K));
}
static inline size_t gq_scl_bytes(int fmt, size_t K, int B) {
  return gq_align256((size_t)B * (gq_kpad(fmt, K) / 32) * 16);
}

// Zero-fills n floats with a kernel (no memset node, so it is safe to capture).
int gq_fill_zero(float *p, size_t n, hipStream_t s);
// INT8 / INT4 rows (K % 32 == 0, gs % 32 == 0) -> T16 Q8_0 / Q4_0, d = fp16(scale *
// head factor); scales and head_scales may be NULL (1.0)
int gq_launch_rows_to_t16(bool int4, const void *b, const float *scales, const float *head_scales, int N, int K, int gs,
                          int head_dim, void *packed, hipStream_t s);
int gq_launch_prep_x(int fmt, const float *x, void *ws, int B, int K, hipStream_t s);

// fp16 batch GEMV (gq_gemv_h.hip)
int gq_gemv_h_min(void);
int gq_gemv_h_plan(int fmt, size_t N, size_t K, int nb, int *R_out, int *ks_out, int *cpw_out);
int gq_gemv_h1_plan(int fmt, size_t N, size_t K, int nb, int *R_out, int *ks_out, int *cpw_out);
// K parts over workgroups (1: the plans above), with the row tiles and waves a
// workgroup then takes
constexpr int kGemvHPartsTw = 4, kGemvHPartsKs = 4;
int gq_gemv_h_parts(int fmt, size_t N, size_t K, int nb);
int gq_launch_gemv_h(int fmt, const void *packed, const float *x, float *y, int N, int K, int nb, hipStream_t s);

// skinny GEMM for M <= 256 (gq_gemv_h.hip); A fp16 in the B fragments' order
// (k_a_to_f16 with the 4-bit permutation for Q4_0 / Q4_K); rs: per-row
// factors applied to C (NULL: none)
int gq_gemm_skinny_plan(int fmt, size_t M, size_t N, size_t K, int *ct_out, int *nck_out);
int gq_launch_gemm_skinny(int fmt, const void *packed, const _Float16 *a16, int lda, void *c, const float *rs,
                          int cbf16, int M, int N, int K, hipStream_t s);

// load-time conversions (gq_loadconv.hip)
int gq_launch_dequant_q6_k(const void *blocks, size_t n_blocks, float *out, int ggml, hipStream_t s);
int gq_launch_f16_to_f32(const void *in, size_t n, float *out, hipStream_t s);

// Library-owned per-device workspace (grown on demand, never shrunk).
int gq_default_workspace(size_t bytes, void **ptr);
// Scratch memory of one call on stream s, for the kernels launched on s in this
// object's lifetime.  Blocks are kept (at most eight a device, of 4 kGqScratchMax bytes
// together; one that is not asked for any more is freed) and pass from call to
// call on one stream, or to another's once the last call's work has ended; a
// call that finds none has memory allocated in its stream's order.  So no call
// waits for another stream or thread, on the host or on the device, and which
// kernels it runs does not depend on them.  ptr is NULL where there is none: more
// than kGqScratchMax asked for, no memory left, or a stream under capture (the
// graph would keep the block's address).
constexpr size_t kGqScratchMax = (size_t)128 << 20;
struct GqScratch {
  void *ptr = nullptr;
  GqScratch(size_t bytes, hipStream_t s);
  ~GqScratch();
  GqScratch(const GqScratch &) = delete;
  GqScratch &operator=(const GqScratch &) = delete;

private:
  hipStream_t stream;
  void *device = nullptr, *block = nullptr;  // (of the kept blocks; none: memory of this call's own)
};
// Q6_K rows of gq_matmul through the tiled GEMM (gq_gemm.hip)
int gq_launch_matmul_q6k(int fmt, const void *packed, const float *a, float *c, size_t M, size_t N, size_t K,
                         hipStream_t s);
// fp16-weight rows of gq_gemm_f16w through the tiled GEMM (gq_gemm.hip)
int gq_launch_gemm_f16w(const void *w, const float *a, float *c, size_t M, size_t N, size_t K, hipStream_t s);
// c[i] = the sum over p of part[p][i], in part order (gq_gemm.hip)
int gq_launch_split_sum(const float *part, float *c, size_t n, int parts, hipStream_t s);
// Compute units of the current device (cached per device; 0 without a device).
int gq_device_cus(void);
