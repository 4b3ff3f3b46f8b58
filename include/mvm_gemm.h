/*
 * mvm_gemm.h -- C ABI of the float32 matrix products of the Mamba block's
 * in_proj and out_proj (libmvm_scan.so).
 *
 * Replaces nn.Linear(d_model, 2 * d_inner) and nn.Linear(d_inner, d_model)
 * of the reference (mlx_vision_mamba/mamba_block.py:125, :153, :165, :191)
 * and their gradients, for all directions of a block at once (:562-566).
 * For each batch index q:
 *
 *   C_q[i, j] = sum_p A_q[i, p] * B_q[p, j] (+ add_q[i, j])    i < m, j < n, p < k
 *
 * Operands are float32; each lies in one of two layouts:
 *   a_kmajor = 1: A_q[i, p] at A[q * a_stride_batch + i * lda + p]
 *   a_kmajor = 0: A_q[i, p] at A[q * a_stride_batch + p * lda + i]
 *   b_kmajor = 1: B_q[p, j] at B[q * b_stride_batch + j * ldb + p]
 *   b_kmajor = 0: B_q[p, j] at B[q * b_stride_batch + p * ldb + j]
 * C_q[i, j] is C[q * c_stride_batch + i * ldc + j], add_q the same of add:
 * NULL, C itself (the products are added to it), or another buffer of C's
 * layout that does not overlap it (a block's residual).  With b_seg > 0 the sum
 * over p runs over segments of b_seg values whose B parts lie b_seg_stride
 * elements apart: p counts as p % b_seg in the addresses above, plus
 * (p / b_seg) * b_seg_stride (the out_proj weights of K directions, each a
 * matrix of its own, in one product over K * d_inner).
 *
 * The products run on the bf16 matrix units with every float32 operand split
 * exactly into three bf16 parts; see csrc/gemm.hip for the error.  Where the
 * split cannot hold the values (infinities, NaN, results to which values below
 * 2^-110 matter) the float32 units compute the tile's part again: the results
 * are float32's, but up to five times slower.  Results are bitwise deterministic.  Conventions are those of mvm_scan.h (status
 * codes, mvm_last_error, caller-owned buffers, host-side validation before
 * any launch, no device allocation).  C must not overlap A or B.
 */
#ifndef MVM_GEMM_H
#define MVM_GEMM_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

typedef struct mvm_gemm_desc {
  int64_t m, n, k;     /* 0..2^30 each */
  int64_t batch;       /* 0..65535 / splits */
  int64_t lda, ldb, ldc;
  int64_t a_stride_batch, b_stride_batch, c_stride_batch;
  int64_t b_seg;        /* 0, or a multiple of 16 that divides k */
  int64_t b_seg_stride;
  int32_t a_kmajor, b_kmajor;  /* 0 or 1 */
  int32_t reserved;    /* must be 0 */
  int32_t splits;      /* parts the sum over p is cut into; 0: chosen by the library */
} mvm_gemm_desc;

/* Validates a descriptor without touching the GPU.  From k = 32 up a k-major
 * operand needs a leading dimension and a batch (and segment) stride that are
 * multiples of 4; leading dimensions are below 2^21.  MVM_ERR_UNSUPPORTED otherwise. */
int mvm_gemm_validate(const mvm_gemm_desc* desc);

/* Bytes of workspace mvm_gemm_f32 needs (0 when the sum is not split). */
int64_t mvm_gemm_workspace_bytes(const mvm_gemm_desc* desc);

/* From k = 32 up k-major operands must be 16-byte aligned; the workspace must
 * be 256-byte aligned.  With k = 0 the products are zero. */
int mvm_gemm_f32(const mvm_gemm_desc* desc, const float* A, const float* B, const float* add,
                 float* C, void* workspace, size_t workspace_bytes, void* stream);

#ifdef __cplusplus
}
#endif

#endif /* MVM_GEMM_H */
