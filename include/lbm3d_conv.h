/*
 * lbm3d_conv.h -- C ABI of the 3-D convolution kernels of liblbm3d.so: BF16
 * implicit-GEMM convolutions on the gfx950 matrix cores (MFMA) with FP32
 * accumulation, forward and backward, for the warm-start surrogate.
 *
 * No reference counterpart: the reference initialises every run at rest
 * (init, Single_phase/LBM_3D_SinglePhase_Solver.py:160-170).  The surrogate
 * predicts steady fields from the geometry and lbm3d_init starts the solver
 * at their equilibrium instead.
 *
 * Layouts (all device pointers, caller-owned; nothing is allocated):
 *   activations  BF16, channels last: x[((b*D + z)*H + y)*W + x][c], for a batch
 *                of `n` volumes of D x H x W voxels and C channels;
 *   weights      BF16 w[co][k], k = tap*cin + ci, tap = (dz+1)*9 + (dy+1)*3 +
 *                (dx+1) for ks = 3 (tap 0 for ks = 1), rows padded with zeros
 *                to kpad = lbm3d_conv_kpad(cin, ks) (a multiple of 32);
 *   bias         FP32 b[cout] (may be NULL);
 *   weight grads FP32 dw[co][kpad].
 * Convolutions are "same" (stride 1, zero padding ks/2, or periodic wrap for
 * the forward convolution with LBM3D_CONV_PERIODIC).  cin and cout must
 * be multiples of 16, at most 256; a batch holds fewer than 2^31 voxels.
 * Activations and BF16 weights start on 16 bytes.
 * Return 0 or a negative LBM3D_E* code (lbm3d.h); lbm3d_conv_last_error()
 * gives the message.
 */
#ifndef LBM3D_CONV_H
#define LBM3D_CONV_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

const char *lbm3d_conv_last_error(void);

/* Padded row length of the weight matrix: ks^3 * cin rounded up to 32. */
int32_t lbm3d_conv_kpad(int32_t cin, int32_t ks);

/* Flags of lbm3d_conv3d_fwd. */
#define LBM3D_CONV_RELU 1     /* apply ReLU to the output */
#define LBM3D_CONV_PERIODIC 2 /* wrap taps past a face to the opposite face instead of zero padding */

/* y = act(conv(x, w) + bias), act = ReLU with LBM3D_CONV_RELU, BF16 out (FP32
 * accumulation); with LBM3D_CONV_PERIODIC each volume is treated as one period
 * of a periodic field (no padding needed around periodic geometries). */
int lbm3d_conv3d_fwd(void *stream, const uint16_t *x, const uint16_t *w, const float *bias, uint16_t *y,
                     int32_t n, int32_t d, int32_t h, int32_t wd, int32_t cin, int32_t cout, int32_t ks,
                     int32_t flags);

/* Fragment order of 3x3x3 weights: BF16 elements of one packed set (cin x cout
 * x 28 tap slots); lbm3d_conv3d_wpack rounds FP32 weights w[cout][kpad] into
 * it for the forward convolution (wp) and, when wt is not NULL, for the data
 * gradient (wt, the flipped weights of lbm3d_conv3d_wflip: a packed convolution
 * from cout to cin channels). */
int64_t lbm3d_conv3d_packed_elements(int32_t cin, int32_t cout);
int lbm3d_conv3d_wpack(void *stream, const float *w, uint16_t *wp, uint16_t *wt, int32_t cin, int32_t cout);
/* The same from BF16 weights. */
int lbm3d_conv3d_wpack_bf16(void *stream, const uint16_t *w, uint16_t *wp, uint16_t *wt, int32_t cin, int32_t cout);
/* Several layers' weights in one go (`layers` is host memory, read during the call). */
typedef struct lbm3d_conv_pack {
  const float *w;
  uint16_t *wp, *wt;
  int32_t cin, cout;
} lbm3d_conv_pack;
int lbm3d_conv3d_wpack_many(void *stream, int32_t count, const lbm3d_conv_pack *layers);

/* lbm3d_conv3d_fwd with ks = 3 and packed weights: the same results, with
 * weight loads that are whole cache lines. */
int lbm3d_conv3d_fwd_packed(void *stream, const uint16_t *x, const uint16_t *wp, const float *bias, uint16_t *y,
                            int32_t n, int32_t d, int32_t h, int32_t wd, int32_t cin, int32_t cout, int32_t flags);

/* lbm3d_conv3d_fwd_packed with ReLU that also writes the 2 x 2 x 2 maximum of y
 * to pool (n volumes of d/2 x h/2 x wd/2 voxels, cout channels; even extents). */
int lbm3d_conv3d_fwd_pool(void *stream, const uint16_t *x, const uint16_t *wp, const float *bias, uint16_t *y,
                          uint16_t *pool, int32_t n, int32_t d, int32_t h, int32_t wd, int32_t cin, int32_t cout,
                          int32_t flags);

/* lbm3d_conv3d_fwd_packed of the concatenation of `low`, upsampled (nearest, by
 * 2: n volumes of d/2 x h/2 x wd/2 voxels, c_low channels), and `skip` (c_skip
 * channels at full extents, all even), which is never built. */
int lbm3d_conv3d_fwd_up(void *stream, const uint16_t *low, const uint16_t *skip, const uint16_t *wp,
                        const float *bias, uint16_t *y, int32_t n, int32_t d, int32_t h, int32_t wd, int32_t c_low,
                        int32_t c_skip, int32_t cout, int32_t flags);
/* Its gradients: the data gradient of the two parts from the flipped packed
 * weights (d_low: BF16 sums over 2 x 2 x 2 blocks of the BF16 gradient at full
 * extents, which is not written), and the weight gradient (workspace of
 * lbm3d_conv3d_wgrad_workspace_bytes for c_low + c_skip channels). */
int lbm3d_conv3d_dgrad_up(void *stream, const uint16_t *dy, const uint16_t *wt, uint16_t *d_low,
                          uint16_t *d_skip, int32_t n, int32_t d, int32_t h, int32_t wd, int32_t c_low,
                          int32_t c_skip, int32_t cout);
int lbm3d_conv3d_wgrad_up(void *stream, const uint16_t *low, const uint16_t *skip, const uint16_t *dy, float *dw,
                          int32_t n, int32_t d, int32_t h, int32_t wd, int32_t c_low, int32_t c_skip, int32_t cout,
                          void *workspace, size_t workspace_bytes);

/* Weights of the data-gradient convolution: wt[ci][tap'*cout + co] =
 * w[co][tap*cin + ci] with tap' = ks^3 - 1 - tap (the kernel flipped and
 * its channel roles swapped), rows padded to lbm3d_conv_kpad(cout, ks). */
int lbm3d_conv3d_wflip(void *stream, const uint16_t *w, uint16_t *wt, int32_t cin, int32_t cout, int32_t ks);

/* dx = conv(dy, wt): the gradient of a convolution's input, given its output
 * gradient dy (BF16, cout channels) and the flipped weights of lbm3d_conv3d_wflip. */
int lbm3d_conv3d_dgrad(void *stream, const uint16_t *dy, const uint16_t *wt, uint16_t *dx, int32_t n,
                       int32_t d, int32_t h, int32_t wd, int32_t cin, int32_t cout, int32_t ks);

/* dw[co][tap*cin + ci] = sum over voxels of dy[v][co] * x[v + off(tap)][ci]
 * (FP32; the padding columns are set to 0), through per-block partial sums in
 * `workspace` of lbm3d_conv3d_wgrad_workspace_bytes() bytes, folded in a fixed
 * order (deterministic). */
size_t lbm3d_conv3d_wgrad_workspace_bytes(int32_t n, int32_t d, int32_t h, int32_t wd, int32_t cin,
                                          int32_t cout, int32_t ks);
int lbm3d_conv3d_wgrad(void *stream, const uint16_t *x, const uint16_t *dy, float *dw, int32_t n, int32_t d,
                       int32_t h, int32_t wd, int32_t cin, int32_t cout, int32_t ks, void *workspace,
                       size_t workspace_bytes);

/* Backward of a fused bias + ReLU: dz = g * (y > 0) elementwise (y the
 * layer's BF16 output; a masked element is g * 0.0 as PyTorch computes it),
 * or dz = g when y is NULL, and db[c] = sum over voxels of dz[v][c] in FP32,
 * through per-block partial sums in `workspace` folded in a fixed order.
 * g, y, dz: [voxels][c] BF16 (dz may be g); c divides 2048, 8..256. */
size_t lbm3d_relu_bias_grad_workspace_bytes(int64_t voxels, int32_t c);
int lbm3d_relu_bias_grad(void *stream, const uint16_t *g, const uint16_t *y, uint16_t *dz, float *db,
                         int64_t voxels, int32_t c, void *workspace, size_t workspace_bytes);

/* lbm3d_relu_bias_grad of a ReLU output y that lbm3d_conv3d_fwd_pool also pooled:
 * the gradient is g plus g_pool shared evenly, in BF16, among the voxels of each
 * 2 x 2 x 2 block that attain its maximum, rounded to BF16.  `share` is scratch
 * of pooled's size; workspace as lbm3d_relu_bias_grad's for n*d*h*w voxels. */
int lbm3d_relu_pool_grad(void *stream, const uint16_t *g, const uint16_t *y, const uint16_t *pooled,
                         const uint16_t *g_pool, uint16_t *dz, float *db, int32_t n, int32_t d, int32_t h, int32_t w,
                         int32_t c, uint16_t *share, void *workspace, size_t workspace_bytes);

/* The network's head: a 1x1x1 convolution from cin to 16 channels, of which the
 * first 4 are used, rounded to BF16 and returned in FP32.  w: the convolution's
 * weights (BF16 w[16][kpad]; rows 0-3 are read), bias its 16 biases (or NULL).
 * out[voxels][4]; or, for the box `core` at `origin` of one volume x of
 * `extents` (3 each, D x H x W), a warm start at once: v[3] = channels 0-2 *
 * scale_v * fluid, rho = 1 + channel 3 * scale_rho * fluid (1 with rho_one), with
 * fluid = solid[voxel of the box] ? 0 : 1. */
int lbm3d_conv_head_fwd(void *stream, const uint16_t *x, const uint16_t *w, const float *bias, float *out,
                        int64_t voxels, int32_t cin);
int lbm3d_conv_head_fields(void *stream, const uint16_t *x, const uint16_t *w, const float *bias, const int8_t *solid,
                           float *rho, float *v, const int32_t extents[3], const int32_t origin[3],
                           const int32_t core[3], int32_t cin, float scale_v, float scale_rho, int rho_one);
/* From the FP32 gradient g[voxels][4] of lbm3d_conv_head_fwd's output: dz[voxels][16],
 * the BF16 gradient of the 16 channels, and db[16], the sums of dz as
 * lbm3d_relu_bias_grad forms them (its workspace, for 16 channels). */
int lbm3d_conv_head_grad(void *stream, const float *g, uint16_t *dz, float *db, int64_t voxels, void *workspace,
                         size_t workspace_bytes);

/* The surrogate's distance input: dist[v] = Euclidean distance from voxel v to
 * the nearest solid voxel (solid[v] != 0) of its volume, with every volume
 * periodic, exact up to `margin` voxels and capped there (also when a volume
 * has no solid).  n volumes of d x h x w voxels, C order; `work` is a float
 * buffer of the same size.  Three separable min-plus passes over offsets
 * |o| <= margin; margin 1..1024. */
int lbm3d_distance_periodic(void *stream, const int8_t *solid, float *dist, float *work, int32_t n, int32_t d,
                            int32_t h, int32_t w, int32_t margin);

/* The surrogate's inputs in one go: per voxel the mask (1 where solid != 0) and
 * the periodic distance divided by `scale` (a power of two), as FP32 pairs
 * out[v][2], or with network != 0 as the first two of 16 BF16 channels
 * out[v][16] (rounded to nearest even, the others zero).  `work` holds
 * 2 * n * d * h * w floats. */
int lbm3d_surrogate_inputs(void *stream, const int8_t *solid, void *out, int network, float scale, float *work,
                           int32_t n, int32_t d, int32_t h, int32_t w, int32_t margin);

#ifdef __cplusplus
}
#endif

#endif /* LBM3D_CONV_H */
