// nn_ops.h -- launchers of the warm-start network's ops (nn_ops.hip).
// Tensors NHWC, activations bf16 (uint16_t bits), parameters fp32.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace cvt {

// 3x3 convolution, padding 1, of N images of H x W pixels:
// out = act(bias + conv(in, w)), Cin and Cout multiples of 32.
struct NnConv {
    // input channels: c0 of in0 (a multiple of 32; at half resolution and
    // upsampled to nearest when up), then Cin - c0 of in1
    const uint16_t *in0;
    int c0, up;
    const uint16_t *in1;
    const uint16_t *w;        // bf16 in the order of nn_weights_bf16
    const float *bias;        // or null
    int relu;
    uint16_t *out;
    uint16_t *pool;           // or null: the 2x2 average of out (H, W even)
    // the first c_low output channels (a multiple of 32) are summed 2x2 into
    // low (H / 2, W / 2, c_low) and out holds the others: the gradient of an
    // input with `up` (H, W even)
    uint16_t *low;
    int c_low;
    // or null: a layer's ReLU output; low (when c_low) or out is zero where
    // it is not positive
    const uint16_t *mask;
};
void nn_conv3x3(hipStream_t s, const NnConv &p, int N, int H, int W, int Cin, int Cout);
// the kernel that it takes for a size: k_conv3x3_keep<8, 2, 2, 1>,
// <4, 2, 2, 1>, <2, 1, 4, 1> and <4, 2, 2, 3>, k_conv3x3<4, 2, 2, 6, 9>,
// <4, 2, 2, 4, 9>, <2, 1, 2, 2, 9>, <4, 2, 2, 2, 3> and <4, 2, 2, 2, 9>
enum NnConvKernel { NN_KEEP_8, NN_KEEP_4, NN_KEEP_2, NN_KEEP_3SLICES, NN_CONV_96, NN_CONV_64,
                    NN_CONV_SMALL, NN_CONV_CIN64, NN_CONV_32, NN_CONV_KERNELS };
int nn_conv3x3_kernel(int N, int H, int W, int Cin, int Cout);
// gradients dw[9][Cout][Cin] and then db[Cout] of the convolution p (its
// inputs) from the out-gradient g; work holds
// nn_dw_max_splits(Cin, Cout) * Cout * (9 * Cin + 1) floats
void nn_conv3x3_dw(hipStream_t s, const NnConv &p, const uint16_t *g, float *dw_db, float *work,
                   int N, int H, int W, int Cin, int Cout);
int nn_dw_max_splits(int Cin, int Cout);
// fp32 weights -> bf16 forward copy and flipped/transposed data-gradient copy
void nn_weights_bf16(hipStream_t s, const float *w, int Cin, int Cout, uint16_t *wf, uint16_t *wb);
// gradient of the 2x2 average
// with mask (a ReLU output shaped as gin), gin = 0 where mask <= 0
void nn_avgpool2_bwd(hipStream_t s, const uint16_t *gout, uint16_t *gin, const uint16_t *mask,
                     int N, int H, int W, int C, int accumulate);
// 1x1 head NN_HEAD_C -> 2 (fp32 out); its backward masks gx by x > 0 (x is a
// ReLU output); dwh_db = [dwh (2C), dbh (2)]; work
// nn_head_splits(M) * (2C + 2) floats
constexpr int NN_HEAD_C = 32;
int nn_head_splits(long M);
void nn_head_fwd(hipStream_t s, const uint16_t *x, const float *wh, const float *bh, float *f,
                 long M);
void nn_head_bwd(hipStream_t s, const uint16_t *x, const float *gf, const float *wh, uint16_t *gx,
                 float *dwh_db, float *work, long M);
// bilinear sample of (nb, R, R, 2) at uv [nb][S][2]; loss partials per 256
// sites; gfield (zeroed by the caller) receives the gradient
void nn_sample_loss(hipStream_t s, const float *field, int R, const float *uv, const float *target,
                    int S, int nb, float scale, float *pred, float *gfield, float *loss_part);
void nn_adam(hipStream_t s, float *w, const float *g, float *m1, float *m2, long n, float lr,
             float b1, float b2, float eps, int t);
#define NN_SUM_BLOCKS 256
// 1 / mean of an n x n density into inv_mean[0] (device), 0 if the sum is 0;
// part is NN_SUM_BLOCKS doubles of scratch
void nn_density_inv_mean(hipStream_t s, const float *rho, int n, double *part, float *inv_mean);
// half-width h of the window that averages the site splat: round(R / sqrt(S))
// - 1, so a window holds about three sites on average
int nn_splat_halfwidth(int R, int S);
// network input (R, R, C) from an n x n density, its 1 / mean (device) and S
// sites (pixel units); count is an R*R float scratch
void nn_prepare(hipStream_t s, const float *rho, int n, const float *inv_mean, const float *xy,
                int S, int R, int C, uint16_t *out, float *count);
// sites += field(site / n) * n for free sites whose target pixel has density
void nn_apply_disp(hipStream_t s, float2 *sites, const uint8_t *fixed, int S, const float *field,
                   int R, const float *rho, int n);

}  // namespace cvt
