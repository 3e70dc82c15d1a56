/*
 * pam_hip_extra.h -- entry points of libpam_hip.so beside the drop-in interface of pam_hip.h: the same computations for
 * callers that have several of them to make at once, or something to learn from one.  Conventions as in pam_hip.h.
 */
#ifndef PAM_HIP_EXTRA_H
#define PAM_HIP_EXTRA_H

#include <stddef.h>

#ifdef __cplusplus
extern "C" {
#endif

/* pam_hip_logsumexp_fwd for a caller that requires finite inputs and wants to know on the host: *nonfinite (a word of page-locked host
 * memory, cleared by the caller) becomes 1 if x holds an infinity or NaN, and `checked` (a hipEvent_t, or NULL) is recorded
 * once that is settled, before the rows' own pass, so that the host can look while the GPU goes on. */
int pam_hip_logsumexp_fwd_finite(const float *x, float *lse, float *log_softmax, float *shift, long rows, long n, float offset,
                                 int *nonfinite, void *checked, void *workspace, size_t workspace_bytes, void *stream);

/* pam_hip_adam_step for `count` tensors with the same scalars, in one launch per 96 of them.  The table is read before the
 * call returns.  Tensors whose p, m or v share memory with another buffer of the list are updated one after the other, in
 * the list's order. */
typedef struct { float *p; const float *g; float *m; float *v; size_t n; } pam_hip_adam_tensor;
int pam_hip_adam_step_many(const pam_hip_adam_tensor *tensors, long count, float beta1, float one_minus_beta1, float beta2,
                           float one_minus_beta2, float eps, float decay, int has_decay, float step_size, float offset,
                           void *stream);

/* a_sums[j] = sum over i of a[i * a_row_stride + j], j < n, and the same for a second matrix of that shape unless b_sums is
 * NULL: ordinary float32 additions in a fixed tree. */
size_t pam_hip_column_sums_workspace_bytes(long rows, long n, int matrices);
int pam_hip_column_sums(const float *a, long a_row_stride, float *a_sums, const float *b, long b_row_stride, float *b_sums,
                        long rows, long n, void *workspace, size_t workspace_bytes, void *stream);

/* Beside pam_hip_gemm_plan: whether the work-groups of that product (exact: of the exact gradient's products) lower their
 * priority as they proceed. */
int pam_hip_gemm_priority_steps(long batch, long m, long n, long k, int exact);

/* How the matrix kernel is launched for that product, with a workspace and operands that are each contiguous along one of
 * their indices: the depth of its k-tiles, the outputs of one work-group and the number of work-groups.  kind: 0 PAM products
 * (of up to four rows without an offset a kernel of their own may run instead), 1 the exact gradient's, 2 a convolution's. */
int pam_hip_gemm_schedule(long batch, long m, long n, long k, int kind, int *k_tile, int *tile_rows, int *tile_columns,
                          long *work_groups);

#ifdef __cplusplus
}
#endif
#endif /* PAM_HIP_EXTRA_H */
