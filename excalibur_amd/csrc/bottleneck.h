// A mobile network's block -- pointwise, depthwise 3x3, pointwise (and a sum) -- in one launch on NHWC halves (bottleneck.hip).
#pragma once
#include "common.h"

struct exhip_bottleneck_layer {  // a pointwise layer of it
    const void* wp;              // the general kernel's packing
    const float* bias;           // or NULL
    long long w_bytes;
    int steps, slab_blocks, channels;  // 32-byte k-steps per pixel, 32-channel blocks per packed slab, output channels
    int runs, start[5];          // runs of k-steps that are summed by themselves and then added, and where they begin
};
struct exhip_bottleneck {
    exhip_bottleneck_layer first, last;
    const void* x;
    const float* slope;          // a PReLU layer behind the first layer, or NULL
    int slope_shared, relu;
    const float *dw_w, *dw_bias, *dw_slope;  // weights [channel][9]; bias, slopes of the PReLU layer behind it, or NULL
    int dw_slope_shared, dw_act;             // activation 0, 1 or 3
    const uint16_t* residual;                // added to the last layer's stored result, or NULL
    uint16_t* y;
    int n, in_h, in_w, out_h, out_w, stride, pad_t, pad_l, pixel_b;  // bytes per input pixel
};
// 0 when launched, EXHIP_ERR_UNSUPPORTED where the layers run by themselves.
int exhip_bottleneck_run(exhip_ctx* ctx, const exhip_bottleneck& b);
