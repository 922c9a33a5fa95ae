// Convolutions on channel-last fp16 copies of their operands (nzhip_conv_cl.hip).
#ifndef NZHIP_CONV_CL_H
#define NZHIP_CONV_CL_H

#include <hip/hip_runtime.h>

#include <cstdint>

namespace nzhip {

enum ClDirection { CL_FORWARD, CL_DATA, CL_WEIGHTS };
// whether a layer (its forward's extents) is within these kernels' extents: 0 not, 1 yes, 2 yes and to be taken (a test says so)
int cl_conv_fits(ClDirection dir, size_t N, size_t C, size_t H, size_t W, size_t O, size_t K_h, size_t K_w, size_t stride, size_t pad, size_t w_batch);
// estimated time in us of one that is
double cl_conv_cost(ClDirection dir, size_t N, size_t C, size_t H, size_t W, size_t O, size_t K_h, size_t K_w, size_t stride, size_t pad, size_t w_batch);
// The three take all their memory before their first launch; NZHIP_E_NOMEM: nothing was launched, and the caller's other ways need less.
// may_keep: a prepared handle of the caller may keep the weights' copy
int cl_conv_forward(float* y, const float* x, const float* w, const float* bias, size_t N, size_t C, size_t H, size_t W, size_t O, size_t K_h,
                    size_t K_w, size_t stride, size_t pad, size_t w_batch, int64_t bias_sp, int64_t bias_sc, int64_t bias_sn, int relu,
                    bool may_keep, hipStream_t s);
int cl_conv_backward_data(float* dx, const float* dy, const float* w, size_t N, size_t C, size_t H, size_t W, size_t O, size_t K_h, size_t K_w,
                          size_t stride, size_t pad, size_t w_batch, int accumulate, hipStream_t s);
int cl_conv_backward_weights(float* dw, const float* x, const float* dy, size_t N, size_t C, size_t H, size_t W, size_t O, size_t K_h, size_t K_w,
                             size_t stride, size_t pad, size_t w_batch, hipStream_t s);

// Convolutions of few tiles in one launch (nzhip_conv_slices.hip). The shape to run one with, -1: not with these
// pixel_bias: a bias that differs from pixel to pixel
int conv_slices_plan(ClDirection dir, size_t N, size_t C, size_t H, size_t W, size_t O, size_t K_h, size_t K_w, size_t stride, size_t pad, size_t w_batch, bool pixel_bias);
int conv_slices_run(bool data, int shape, float* y, const float* x, const float* w, const float* bias, size_t N, size_t C, size_t H, size_t W, size_t O, size_t K_h, size_t K_w,
                    size_t stride, size_t pad, size_t w_batch, int64_t bias_sp, int64_t bias_sc, int64_t bias_sn, int relu, int accumulate, hipStream_t s);

}  // namespace nzhip

#endif
