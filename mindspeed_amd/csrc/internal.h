// Entry points for this package's own use only: combinations of what include/mindspeed_amd.h declares that save a
// launch, and a diagnostic.  Not part of the C ABI that ms_version() stands for.
#pragma once

#include "../../include/mindspeed_amd.h"

#ifdef __cplusplus
extern "C" {
#endif

/* The hash of these declarations and of those in mindspeed_amd.h that the library was built from (build.py: interface_hash):
 * what a binding that passes arguments by them compares with its own before its first call. */
const char *msi_interface(void);
/* ms_moe_routing_map_permute and ms_moe_routing_map_probs in one: permuted_probs [num_rows] in the dtype of probs (both may
 * be NULL) and sorted_token_ids [num_rows] (may be NULL) are written beside the rows; rows that no map entry leads to get
 * zeros.  Without tokens neither may be asked for. */
int msi_routing_map_permute(ms_stream_t stream, const void *tokens, const void *routing_map, int64_t num_tokens,
                            int64_t num_experts, int64_t hidden, int dtype, int64_t num_rows, int drop_and_pad,
                            void *permuted, int32_t *row_id_map, int32_t *sorted_flat, int64_t *tokens_per_expert,
                            const void *probs, int probs_dtype, void *permuted_probs, int64_t *sorted_token_ids,
                            void *workspace, size_t workspace_bytes);
/* ms_moe_token_unpermute_grad, and rows r of grad_permuted with sorted_flat[r] < 0 (may be NULL) written as zeros
 * (ms_moe_zero_unmapped_rows). */
int msi_unpermute_grad(ms_stream_t stream, const void *permuted_tokens, const void *grad_unpermuted,
                       const int32_t *row_id_map, const void *probs, int probs_dtype, int64_t num_tokens, int64_t topk,
                       int64_t hidden, int dtype, int64_t num_rows, const int32_t *sorted_flat, void *grad_permuted,
                       void *grad_probs);
/* Both gradients of one grouped matmul y = x w (split on rows): dx [m, k] = grad w^T and dw [num_groups, k, n] = x^T grad (fp32
 * with accumulate: added to), the two ms_gmm calls of the backward pass in one.  grad [m, n], x [m, k], weight [num_groups, k, n]
 * by strides; dx and dw contiguous. */
int msi_gmm_backward_workspace_size(int64_t num_groups, int64_t m, int64_t k, int64_t n, int dtype, int dw_dtype,
                                    int accumulate, size_t *bytes);
int msi_gmm_backward(ms_stream_t stream, const void *grad, int64_t grad_stride0, int64_t grad_stride1, const void *x,
                     int64_t x_stride0, int64_t x_stride1, const void *weight, int64_t w_stride_group, int64_t w_stride0,
                     int64_t w_stride1, void *dx, void *dw, const int64_t *group_list, int group_list_type,
                     int64_t num_groups, int64_t m, int64_t k, int64_t n, int dtype, int dw_dtype, int accumulate,
                     void *workspace, size_t workspace_bytes);
/* Diagnostic, host only: whether a 16-bit launch split on rows with these group sizes (a host array) gives every XCD
 * consecutive tiles of the whole launch instead of an eighth of every group's, by the rule of the lookup in the group list
 * (from_list != 0) or of the schedule kernel's table; num_cus: the GPU's compute units.  Evaluates the functions the kernels
 * call, so a test can check that a launch takes the order it is meant to: a launch of its own, not dX in the launch of both
 * gradients, where more groups share the rows of their last tiles.  (A table falls back to eighths where shares equal
 * in cost need more workgroups than the launch has, and makes no such shares where it deals out whole groups.) */
int msi_gmm_takes_together(const int64_t *rows, int64_t num_groups, int64_t k, int64_t n, int from_list, int num_cus,
                           int *together);

#ifdef __cplusplus
}
#endif
