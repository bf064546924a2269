/*
 * megagemm_hip_fused.h -- entry points that do in one launch what takes several through
 * megagemm_hip.h, for the calls whose time is launches and latency: RMSNorm backward of a few rows,
 * and the two projections of the SwiGLU block (reference: megagemm/swiglu.py:165-172, two
 * torch.matmul around the Triton activation) in a decoding step of a small batch -- and the activation
 * where no backward pass follows.
 * Conventions as in megagemm_hip.h.
 */
#ifndef MEGAGEMM_HIP_FUSED_H
#define MEGAGEMM_HIP_FUSED_H

#include "megagemm_hip.h"

#ifdef __cplusplus
extern "C" {
#endif

/*
 * 1 if mg_rmsnorm_bwd_small takes this shape (and is the faster way there), else 0.  0 as well while any
 * mg_set_option override is in force that mg_rmsnorm_bwd follows ("force_generic", "bwd_*", "narrow_groups",
 * "xcd_group"), so that a caller who asks first gets the backward pass the override is about.
 */
int mg_rmsnorm_bwd_small_fits(int64_t rows, int64_t cols, int dtype);

/*
 * RMSNorm backward as mg_rmsnorm_bwd followed by mg_rmsnorm_dw_reduce, without a workspace: dx and
 * the finished dW (in fp32, in `dtype`, both, or -- both NULL -- neither).  Summation order of dW is
 * fixed, but not that of the two-call path.  Shapes it does not take: MG_ERR_UNSUPPORTED.
 * No output may overlap an input: unlike in the two calls, dx is written while x and dy of the same rows are
 * still read for dW, and dW while w and inv_rms are read for dx.  Such a call is refused (MG_ERR_INVALID_ARG).
 */
int mg_rmsnorm_bwd_small(void* dx, float* dw_f32, void* dw_cast, const void* dy, const void* x, const void* w,
                         const float* inv_rms, int64_t rows, int64_t cols, int dtype, void* stream);

/* Most rows (tokens) the two entry points below take. */
#define MG_BLOCK_MAX_TOKENS 64

/*
 * h[t, n] = silu(g) * u with g = sum_k x[t, k] * w12[n, k], u = sum_k x[t, k] * w12[hidden + n, k]:
 * first projection and activation in one pass, g and u kept in fp32.
 *   h   [tokens, hidden], x [tokens, d_model], w12 [2 * hidden, d_model]
 *   dtype  MG_F16 or MG_BF16; 1 <= tokens <= MG_BLOCK_MAX_TOKENS; d_model a multiple of 8;
 *   x and w12 16-byte aligned; h overlaps neither.  Anything else: MG_ERR_UNSUPPORTED or MG_ERR_INVALID_ARG.
 */
int mg_block_gate_up(void* h, const void* x, const void* w12, int64_t tokens, int64_t d_model, int64_t hidden,
                     int dtype, void* stream);

/*
 * out[t, n] = sum_k h[t, k] * w3[n, k]: the second projection.
 *   out [tokens, d_model], h [tokens, hidden], w3 [d_model, hidden]; hidden a multiple of 8; otherwise as above.
 */
int mg_block_down(void* out, const void* h, const void* w3, int64_t tokens, int64_t d_model, int64_t hidden,
                  int dtype, void* stream);

/*
 * mg_swiglu_fwd for an input that no backward pass will read again: the same results; gu is read past the
 * memory-side cache and leaves the room in it to others (mg_swiglu_fwd keeps up to 128 MiB of it there).
 */
int mg_swiglu_fwd_only(void* h, const void* gu, int64_t M, int64_t H, int dtype, void* stream);

#ifdef __cplusplus
}
#endif

#endif /* MEGAGEMM_HIP_FUSED_H */
