/*
 * megagemm_hip_mlp.h -- the whole SwiGLU block (reference: megagemm/swiglu.py:165-172, two torch.matmul
 * around the Triton activation, and their autograd) on this library's own matrix products, with the activation
 * and its backward inside them: forward in two launches, backward in two, and one more for each
 * product whose k is split.
 * Conventions as in megagemm_hip.h.  x, out, dy, dx [tokens, d_model]; w12 [2 * hidden, d_model], gate rows first;
 * w3 [d_model, hidden]; gate_up [tokens, 2 * hidden]; h [tokens, hidden]; all of `dtype`, MG_F16 or MG_BF16.
 */
#ifndef MEGAGEMM_HIP_MLP_H
#define MEGAGEMM_HIP_MLP_H

#include "megagemm_hip.h"

#ifdef __cplusplus
extern "C" {
#endif

/*
 * 1 if the two entry points below take these sizes: d_model and hidden multiples of 64 and at most 65536, at least one
 * token, every tensor below 2 GiB.  Not a statement about speed.
 */
int mg_mlp_fits(int64_t tokens, int64_t d_model, int64_t hidden, int dtype);

/* What a call of the block consists of: forward and backward, forward alone, or forward and a backward pass for dx alone. */
#define MG_MLP_ALL 0
#define MG_MLP_FORWARD_ONLY 1
#define MG_MLP_X_LEARNS 2

/*
 * 1 where they are also taken rather than library products around mg_swiglu_fwd and mg_swiglu_bwd (0 for sizes they do not
 * take) in such a call.  A rule fitted to times of both sides, which stand beside it: the few sizes it gets wrong lose a few per cent.
 * Both bindings ask this.
 */
int mg_mlp_preferred(int64_t tokens, int64_t d_model, int64_t hidden, int dtype, int call);

/* What a workspace is for: the forward pass, or a backward pass that wants the sum of these. */
#define MG_MLP_FORWARD 0
#define MG_MLP_DX 1
#define MG_MLP_DW12 2
#define MG_MLP_DW3 4

/*
 * Bytes of workspace a pass needs on the current device, 0 for none: where a product has few tiles, its k is split over workgroups,
 * whose sums meet there in fp32.  For sizes mg_mlp_preferred takes at most about 260 MiB, and less than the tensors the pass writes.
 */
int mg_mlp_workspace(int64_t tokens, int64_t d_model, int64_t hidden, int dtype, int pass, int64_t* bytes);

/*
 * [gate | up] = x * w12^T, h = silu(gate) * up from sums kept in fp32, out = h * w3^T.
 * gate_up may be NULL where no backward pass follows, workspace where none is needed.  Pointers 16-byte aligned; no output
 * (the workspace is one) overlaps an input or another output.  MG_ERR_UNSUPPORTED for sizes mg_mlp_fits does not take.
 */
int mg_mlp_fwd(void* out, void* h, void* gate_up, const void* x, const void* w12, const void* w3, void* workspace, int64_t workspace_bytes,
               int64_t tokens, int64_t d_model, int64_t hidden, int dtype, void* stream);

/*
 * The gradients for dy as the gradient of out: dx, dw12 and dw3, each NULL where not wanted.  gate_up and h as
 * mg_mlp_fwd left them.  d_gate_up [tokens, 2 * hidden] is written unless dx and dw12 are both NULL (it may then be NULL).
 * An input that no wanted gradient reads may be NULL: x without dw12, w12 without dx, w3 and gate_up without both, h without dw3.
 * Sums in a fixed order: bit-identical from run to run.  Otherwise as mg_mlp_fwd.
 */
int mg_mlp_bwd(void* dx, void* dw12, void* dw3, void* d_gate_up, const void* dy, const void* x, const void* w12, const void* w3,
               const void* gate_up, const void* h, void* workspace, int64_t workspace_bytes, int64_t tokens, int64_t d_model, int64_t hidden,
               int dtype, void* stream);

#ifdef __cplusplus
}
#endif

#endif /* MEGAGEMM_HIP_MLP_H */
