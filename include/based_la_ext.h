/*
 * based_la_ext.h -- further entry points of libbased_la.so (based_la.h): states on the segment-state
 * chunked shapes, and the parallel kernel on strided tensors.  Conventions, status codes and argument
 * rules are based_la.h's.  No reference counterparts.
 *
 * States.  la_based_chunked_fwd exports and imports states itself for bf16, d = 16, dv <= 64; for the other
 * bf16 shapes (d <= 64, dv <= 128) these calls do, beside la_based_chunked_fwd_num_den.  States are
 * fp32 (B, H, F, dv + 1) = [sum_u phi(a k_u) v_u^T | sum_u phi(a k_u)], F = 1 + d + d (d + 1) / 2, in
 * the feature order of taylor_feature_map (benchmarks/chunked_attention_benchmark.py:34-53), with
 * a = (scale^2 d)^(1/4), so that phi(a q) . phi(a k) = 1 + s + s^2 / 2 for s = scale q.k.
 */
#ifndef BASED_LA_EXT_H
#define BASED_LA_EXT_H

#include <stddef.h>

#ifdef __cplusplus
extern "C" {
#endif

/* Scratch enough for either call (0 for shapes outside them); 16-byte aligned. */
size_t la_based_state_workspace_bytes(int B, int H, int N, int d, int dv);

/* state_out = state_in (zero if NULL) + these tokens' state.  state_in may be state_out.
 * N = 0 writes nothing. */
int la_based_state_export(const void* k, const void* v, int in_dtype, const float* state_in_or_null,
                          float* state_out, int B, int H, int N, int d, int dv, float scale,
                          void* workspace, size_t workspace_bytes, void* hip_stream);

/* out = (num + phi(a q) S) / (den + phi(a q) z + eps) for state = [S | z] (the numerator with
 * normalize = 0); num, den as la_based_chunked_fwd_num_den gives them.  out may be num when
 * out_dtype is LA_F32. */
int la_based_state_apply(const void* q, int in_dtype, const float* state, const float* num,
                         const float* den, void* out, int out_dtype, int B, int H, int N, int d, int dv,
                         float scale, float eps, int normalize, void* workspace,
                         size_t workspace_bytes, void* hip_stream);

/*
 * la_based_parallel_fwd on tensors whose heads lie in a token's row, such as the (B, N, 3, H, d)
 * output of a fused q/k/v projection and the (B, N, H dv) input of the next one: element (b, h, t, i)
 * of x lies at x + b x_strides[0] + h x_strides[1] + t x_strides[2] + i (strides in elements, in that
 * order, >= 0 and multiples of 8; tensors 16-byte aligned: LA_ERR_BAD_ALIGNMENT otherwise).  k_strides also serve q.
 * bf16 in and out, normalised; shapes of the ring-copy kernel (d % 8 == 0, d <= 64, dv % 8 == 0,
 * dv <= 128, N > 64) that la_based_parallel_fwd runs on it, LA_ERR_UNSUPPORTED_DIM for others (the
 * caller copies then).  workspace: la_based_parallel_workspace_bytes bytes.
 */
int la_based_parallel_fwd_strided(const void* q, const void* k, const void* v, void* out, int B, int H,
                                  int N, int d, int dv, const long long* k_strides,
                                  const long long* v_strides, const long long* out_strides, float scale,
                                  float eps, void* workspace, size_t workspace_bytes, void* hip_stream);

/* The workspace of la_based_parallel_fwd_strided (that of la_based_parallel_fwd), 0 for sizes and strides that
 * it does not take: a caller that would then copy asks before it allocates an output. */
size_t la_based_parallel_strided_workspace_bytes(int B, int H, int N, int d, int dv, const long long* k_strides,
                                                 const long long* v_strides, const long long* out_strides);

#ifdef __cplusplus
}
#endif

#endif /* BASED_LA_EXT_H */
