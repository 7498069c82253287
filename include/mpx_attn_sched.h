/*
 * Schedule entries of libmpx_attn.so beside mpx_attn.h: variants of its calls
 * whose caller sizes the workspace for one schedule. Conventions (return
 * codes, strides, streams) are those of mpx_attn.h.
 */
#ifndef MPX_ATTN_SCHED_H
#define MPX_ATTN_SCHED_H

#include "mpx_attn.h"

#ifdef __cplusplus
extern "C" {
#endif

/*
 * mpx_attn_bwd_dropout (dropout_p = 0: mpx_attn_bwd) on the recomputing
 * schedule, for grouped K/V heads: with a workspace of at least
 * mpx_attn_bwd_grouped_workspace_bytes(...) bytes the query heads of a K/V
 * head are cut into parts that run as separate workgroups and leave float32
 * sums in the workspace, added up and rounded once by a last kernel; with less
 * (mpx_attn_bwd_workspace_bytes at least) each group is one part. No
 * counterpart in the reference, whose flash_attention takes equal head counts
 * (mlx_primitives/attention/flash.py:151-154).
 */
size_t mpx_attn_bwd_grouped_workspace_bytes(int B, int H, int H_kv, int Sq, int Sk, int D,
                                            int dtype, int window_left);

int mpx_attn_bwd_grouped(const void* q, const void* k, const void* v, const void* o,
                         const void* dout, const float* lse, void* dq, void* dk, void* dv,
                         const int64_t* q_strides, const int64_t* k_strides,
                         const int64_t* v_strides, const int64_t* o_strides,
                         const int64_t* do_strides, const int64_t* dq_strides,
                         const int64_t* dk_strides, const int64_t* dv_strides,
                         int B, int H, int H_kv, int Sq, int Sk, int D, float scale, int causal,
                         int window_left, int window_right, int dtype, float dropout_p,
                         uint64_t seed, void* workspace, size_t workspace_bytes, void* stream);

/*
 * The same call on the stored-dS schedule (mpx_attn_bwd_ds_workspace_bytes),
 * whatever its size: MPX_EINVAL where the problem has none or the workspace
 * does not hold it.
 */
int mpx_attn_bwd_stored(const void* q, const void* k, const void* v, const void* o,
                        const void* dout, const float* lse, void* dq, void* dk, void* dv,
                        const int64_t* q_strides, const int64_t* k_strides,
                        const int64_t* v_strides, const int64_t* o_strides,
                        const int64_t* do_strides, const int64_t* dq_strides,
                        const int64_t* dk_strides, const int64_t* dv_strides,
                        int B, int H, int H_kv, int Sq, int Sk, int D, float scale, int causal,
                        int window_left, int window_right, int dtype, float dropout_p,
                        uint64_t seed, void* workspace, size_t workspace_bytes, void* stream);

/*
 * 1 when the dropout backward runs faster on the stored-dS schedule
 * (mpx_attn_bwd_dropout with mpx_attn_bwd_ds_workspace_bytes) than recomputing
 * (mpx_attn_bwd_grouped for grouped heads), else 0: launches that do not fill
 * the chip, where mpx_attn_bwd_dropout recomputes whatever the workspace holds,
 * and grouped heads that mpx_attn_bwd_grouped runs in parts (which
 * mpx_attn_bwd_dropout does not: with that workspace it stores dS).
 */
int mpx_attn_bwd_ds_preferred(int B, int H, int H_kv, int Sq, int Sk, int D, int dtype,
                              int window_left);

/*
 * mpx_attn_fwd_rope with K rotated inside the kernel as well: k as given, its
 * row j at position k_offset + j (the bits of mpx_rope applied to k first, then
 * mpx_attn_fwd_rope). bfloat16 inputs, 16-bit tables, D = 128; q_offset + Sq and
 * k_offset + Sk at most n_pos. Workspace: mpx_attn_fwd_workspace_bytes.
 * Replaces both sides of the reference's fused kernel
 * (mlx_primitives/kernels/fused_rope_attention.py:766-800).
 * Available where the launch runs in key groups (calls that leave CUs empty;
 * elsewhere MPX_EUNSUPPORTED). _preferred: 1 where it is, and is faster than a
 * pass over K.
 */
int mpx_attn_fwd_rope_qk_preferred(int B, int H, int Sq, int Sk, int D, int causal,
                                   int window_left, int window_right, int dtype, int cache_dtype);

int mpx_attn_fwd_rope_qk(const void* q, const void* k, const void* v, void* o,
                         const int64_t* q_strides, const int64_t* k_strides,
                         const int64_t* v_strides, const int64_t* o_strides,
                         int B, int H, int H_kv, int Sq, int Sk, int D, float scale, int causal,
                         int window_left, int window_right, int dtype,
                         const void* cos_cache, const void* sin_cache, int q_offset, int k_offset,
                         int n_pos, int cache_dtype, void* workspace, size_t workspace_bytes,
                         void* stream);

/*
 * How a forward call of this size runs, for tests and tuning: *key_groups is
 * the number of key groups that a workgroup's waves are cut into (1, 2 or 4),
 * *splits the most ranges that a query tile's keys are split into (1: none),
 * *balanced 1 where two workgroups per CU take long and short query tiles
 * together. block_size > 0: paged prefill over tables of Sk tokens (no window)
 * with pages of that size, `alibi` != 0 with ALiBi slopes. D as the kernels
 * take it. MPX_EINVAL for empty sizes. No counterpart in the reference.
 */
int mpx_attn_fwd_form(int B, int H, int Sq, int Sk, int D, int causal, int window_left,
                      int window_right, int dtype, int block_size, int alibi, int* key_groups,
                      int* splits, int* balanced);

#ifdef __cplusplus
}
#endif

#endif /* MPX_ATTN_SCHED_H */
