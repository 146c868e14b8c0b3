/* fwn_rows.h - C ABI of the row permutation passes either side of the mesh transformer's layer
 * loop, fused with the layer norms next to them (same library as fwn_attn.h).
 *
 * The reference sorts the mesh nodes along a Hilbert curve so that the k-hop mask has fewer
 * live tiles: it gathers the node features with the permutation before the 24 layers and
 * scatters them back after the final norm (patch.py:274-276, 288-292). Each of those is one
 * extra pass over [batch, n, channels] per step. Here the gather is fused with the first
 * block's layer norm and the scatter with the final layer norm and its per-member affine, so
 * the permutation costs no pass of its own.
 *
 * Conventions (as in fwn_attn.h): status codes and fwn_last_error(); launchers validate on the
 * host, enqueue on `stream`, allocate nothing and keep no pointer. Tensors are contiguous
 * [batch, n, channels] in the dtype of the descriptor; statistics are computed in float32.
 * `perm` is a device array of n int64 that must be a permutation of 0..n-1. An entry outside
 * [0, n) yields a zero row (gather) or is dropped (scatter); repeated entries make the scatter
 * write one row twice in an unspecified order. Neither touches memory outside the tensors.
 */
#ifndef FWN_ROWS_H_
#define FWN_ROWS_H_

#include <stdint.h>

#include "fwn_attn.h"

#ifdef __cplusplus
extern "C" {
#endif

#define FWN_ROWS_MAX_CHANNELS 4096

typedef struct fwn_rows_desc {
  int32_t batch;
  int32_t n;         /* rows (mesh nodes) per batch member */
  int32_t channels;  /* features per row: a multiple of 8, at most FWN_ROWS_MAX_CHANNELS */
  int32_t dtype;     /* fwn_dtype of x and of every output */
  float eps;         /* layer-norm epsilon, added to the biased variance */
} fwn_rows_desc;

/* x_out[b, i, :] = x[b, perm[i], :] and, when norm_out is not NULL,
 * norm_out[b, i, :] = (x_out[b, i, :] - mean) / sqrt(var + eps) over the channels (a layer norm
 * without scale or offset). Replaces jnp.take(node_features, perm, axis=1) before the layer
 * loop (patch.py:274-276) fused with the first block's st.layernorm(x, create_scale=False,
 * create_offset=False) (patch.py:244). x and x_out must not overlap. */
int fwn_rows_gather_norm_launch(const fwn_rows_desc* d, const void* x, const int64_t* perm,
                                void* x_out, void* norm_out, void* stream);

/* out[b, perm[i], :] = layer_norm(x[b, i, :]) * mul[b, :] + add[b, :], with mul and add float32
 * [batch, channels] (NULL means 1 and 0). Replaces the final st.layernorm, the per-member
 * affine that LinearNormConditioning applies to it (its scale and offset come from the
 * conditioning vector, computed by the caller) and jnp.take(x, argsort(perm), axis=1)
 * (patch.py:288-292). x and out must not overlap. */
int fwn_rows_norm_scatter_launch(const fwn_rows_desc* d, const void* x, const int64_t* perm,
                                 const float* mul, const float* add, void* out, void* stream);

/* out[b, i, :] = layer_norm(x[b, i, :]) * mul[b, :] + add[b, :] (mul and add float32
 * [batch, channels], NULL meaning 1 and 0): the block's conditioned layer norm in one pass, the
 * fwn_rows_norm_scatter_launch pass without a permutation. Replaces
 * norm_conditioning_layer(st.layernorm(x, create_scale=False, create_offset=False)) in front of
 * the attention and of the feed-forward of every block (patch.py:240-244, 250-251), whose
 * LinearNormConditioning scale and offset the caller evaluates from the conditioning vector.
 * x and out must not overlap. */
int fwn_rows_norm_affine_launch(const fwn_rows_desc* d, const void* x, const float* mul,
                                const float* add, void* out, void* stream);

/* sum[b, i, :] = x[b, i, :] + y[b, i, :] (added in float32, rounded once to the dtype) and
 * out[b, i, :] = layer_norm(sum[b, i, :]) * mul[b, :] + add[b, :]: the block's residual add
 * fused with the conditioned layer norm that reads its result. Replaces `x = x + mha(...)`
 * followed by the feed-forward's norm_conditioning_layer(st.layernorm(x)), and the feed-forward
 * residual followed by the next block's conditioned layer norm (patch.py:240-253). sum may be x
 * or y itself (an in-place residual update) or disjoint from both; out must not overlap x, y or
 * sum. */
int fwn_rows_add_norm_affine_launch(const fwn_rows_desc* d, const void* x, const void* y,
                                    const float* mul, const float* add, void* sum, void* out,
                                    void* stream);

/* The conditioning of `count` (1 to FWN_COND_MAX) norms from one conditioning vector: for norm l, with
 * weight[l] a contiguous [2 * channels, cond_size] matrix and bias[l] of 2 * channels entries, both
 * in `dtype` as cond [batch, cond_size],
 *   mul[l, b, c] = 1 + weight[l][c, :] . cond[b, :] + bias[l][c]
 *   add[l, b, c] = weight[l][channels + c, :] . cond[b, :] + bias[l][channels + c]
 * in float32, the affine the norm passes take (LinearNormConditioning's projections, which the
 * reference evaluates norm by norm, patch.py:240-253, 288-292). mul and add are float32 [count,
 * batch, channels]. weight and bias are host arrays of device pointers, read before returning. */
#define FWN_COND_MAX 64
int fwn_cond_affine_launch(int32_t count, int32_t batch, int32_t channels, int32_t cond_size, int32_t dtype,
                           const void* cond, const void* const* weight, const void* const* bias, float* mul,
                           float* add, void* stream);

/* Backward of the passes above: for every row i of x (the rows a pass normalised, with xhat their
 * layer norm and rstd its 1 / sqrt(var + eps), recomputed from x),
 *
 *   g[b, i, :]  = rstd (gm - mean(gm) - xhat mean(gm xhat)) + g_res[b, i, :],  gm = g_norm mul
 *   g_mul[b, :] = sum over i of g_norm xhat,   g_add[b, :] = sum over i of g_norm
 *
 * computed in float32; g is written to gx in the dtype. g_norm (NULL: zeros) is the gradient of
 * the norm's output, g_res (NULL: zeros) that of the sum or copy x itself also went to, mul as in
 * the forward (NULL: 1). g_mul and g_add (float32 [batch, channels]) are written when both are
 * non-NULL; that needs fwn_rows_norm_bwd_workspace_size bytes of workspace (16-byte aligned), used
 * until the launch's stream work is done, and none otherwise. The sums run in a fixed order.
 * With perm, `perm_rows` says what it permutes:
 *   FWN_ROWS_PERM_GRAD: row i's g_norm is row perm[i] of the tensor (backward of norm_scatter);
 *   FWN_ROWS_PERM_OUT: g is written to row perm[i] of gx (backward of gather_norm).
 * Entries of perm outside [0, n) read a zero row or drop the row. gx must not overlap the inputs. */
#define FWN_ROWS_PERM_GRAD 1
#define FWN_ROWS_PERM_OUT 2
int fwn_rows_norm_bwd_workspace_size(const fwn_rows_desc* d, uint64_t* bytes);
int fwn_rows_norm_bwd_launch(const fwn_rows_desc* d, const void* x, const int64_t* perm, int32_t perm_rows,
                             const void* g_norm, const void* g_res, const float* mul, void* gx, float* g_mul,
                             float* g_add, void* workspace, uint64_t workspace_bytes, void* stream);

/* dw[o, i] = sum over r of g[r, o] * x[r, i] and, where db is given, db[o] = sum over r of g[r, o]:
 * the gradients of y = x w^T + b with respect to w and b, as the transformer block's projections and
 * feed-forward take them (patch.py:165-177, 233-253). g is [rows, outs], x [rows, ins], dw [outs, ins],
 * db [outs], all contiguous bfloat16, 16-byte aligned; sums are float32, rounded to bfloat16 once.
 * outs and ins are positive multiples of FWN_LINEAR_UNIT, each at most FWN_LINEAR_MAX; rows >= 1.
 * The workspace (fwn_linear_wgrad_workspace_size bytes, 16-byte aligned) holds float32 partial sums;
 * its contents before the call do not matter. */
#define FWN_LINEAR_UNIT 64
#define FWN_LINEAR_MAX 16384
int fwn_linear_wgrad_workspace_size(int64_t rows, int32_t outs, int32_t ins, uint64_t* bytes);
int fwn_linear_wgrad_launch(int64_t rows, int32_t outs, int32_t ins, const void* g, const void* x, void* dw, void* db,
                            void* workspace, uint64_t workspace_bytes, void* stream);

#ifdef __cplusplus
}  /* extern "C" */
#endif

#endif /* FWN_ROWS_H_ */
