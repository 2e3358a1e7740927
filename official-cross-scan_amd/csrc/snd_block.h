// The passes of a VSS block around its scan (snd_block.hip), as the PyTorch extension launches them.  Not part of the C ABI
// of include/snd_scan.h.  Activations have the type `dtype` (SND_F32 / SND_F16 / SND_BF16); parameters and the gradients
// of parameters are fp32, the latter accumulated into (the caller clears them).  All return an snd_status.
#pragma once
#include "snd_scan.h"

#define SND_BLOCK_MAX_NORM 1024                    /* channels of snd_block_norm */
#define SND_BLOCK_MAX_RANK 64                      /* dt rank */

extern "C" {
typedef struct {
    int32_t batch, nrows, ncols, inner;            /* inner: channels of the scan's feature map */
    int32_t n_groups, dstate, rank, dtype;
} snd_block_shape;

/* LayerNorm over the last of [tokens, channels]; stats (mean, 1 / std per token) is written if not null. */
int snd_block_norm_fwd(const void *x, int x_dtype, const float *gamma, const float *beta, float eps, int64_t tokens, int channels,
                       void *y, int y_dtype, float *stats, snd_stream_t stream);
int snd_block_norm_bwd(const void *dy, int dy_dtype, const void *x, int x_dtype, const float *gamma, const float *stats, int64_t tokens,
                       int channels, void *dx, float *dgamma, float *dbeta, snd_stream_t stream);

/* A = -exp(A_logs) (nA values); w = wx [rows, cols] in `dtype` and (if not null) its transpose wt. */
int snd_block_params(const float *A_logs, int nA, const float *wx, int rows, int cols, int dtype, float *A, void *w, void *wt, snd_stream_t stream);

/* Depthwise 3x3 convolution + bias + SiLU: x = the first `inner` channels of xz [batch, nrows, ncols, 2 * inner] ->
 * u [batch, inner, nrows, ncols]; pre (may be null): the value before SiLU.  Backward: du -> the first half of dxz. */
int snd_block_conv_fwd(const snd_block_shape *s, const void *xz, const float *w, const float *bias, void *pre, void *u, snd_stream_t stream);
int snd_block_conv_bwd(const snd_block_shape *s, const void *du, const void *pre, const void *xz, const float *w, void *dxz, float *dw,
                       float *dbias, snd_stream_t stream);

/* LayerNorm over the channels of y [batch, inner, nrows, ncols] (fp32) times SiLU(z), z = the second half of xz ->
 * out [batch, nrows, ncols, inner].  Backward: dout -> dy (fp32) and the second half of dxz. */
int snd_block_gate_fwd(const snd_block_shape *s, const float *y, const void *xz, const float *gamma, const float *beta, float eps, void *out,
                       float *stats, snd_stream_t stream);
int snd_block_gate_bwd(const snd_block_shape *s, const void *dout, const float *y, const void *xz, const float *gamma, const float *beta,
                       const float *stats, float *dy, void *dxz, float *dgamma, float *dbeta, snd_stream_t stream);

/* proj [batch, n_groups, rank + 2 * dstate, nrows * ncols]: delta[b, g, d] = sum_r w[g, d, r] * proj[b, g, r]
 * (delta [batch, n_groups * inner, nrows * ncols]).  Backward: dproj = [w^T ddelta | dB | dC]. */
int snd_block_dt_fwd(const snd_block_shape *s, const void *proj, const float *w, void *delta, snd_stream_t stream);
int snd_block_dt_bwd(const snd_block_shape *s, const void *ddelta, const void *dB, const void *dC, const float *w, void *dproj, snd_stream_t stream);

/* out[g][m][n] += sum over batch images b and pixels p of a[b, g, m, p] * c[b, g, n, p]; strides in elements. */
int snd_block_wgrad(const void *a, int64_t a_batch, int64_t a_group, const void *c, int64_t c_batch, int64_t c_group, int batch, int groups,
                    int M, int N, int64_t pixels, int dtype, float *out, snd_stream_t stream);
/* The weight and (if not null) bias gradient of a linear layer: dw[m][n] += sum over tokens of dy[t][m] * x[t][n], dbias[m] +=
 * sum of dy[t][m]; dy [tokens, M], x [tokens, N] of a 16-bit type, M and N even. */
int snd_block_linear_wgrad(const void *dy, const void *x, int64_t tokens, int M, int N, int dtype, float *dw, float *dbias, snd_stream_t stream);
}
