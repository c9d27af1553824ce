// What the float32 convolution kernels (conv_f32.hip, conv_f32_thirds.hip) share: a launch's parameters and the epilogue of a few channels
// per lane.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "common.h"

namespace {

typedef exhip_v4i v4i;
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));

constexpr unsigned kRsrcWord3 = 0x00020000u;      // raw buffer: out-of-range loads return 0, such stores are dropped
constexpr unsigned kOutOfRange = 0xfffff000u;     // a lane offset beyond every view
constexpr int kMaxSplit = 8;

// How a step's 32 bytes lie in the input: kPoint one tap, always inside the image (1x1 filters without padding); kTaps 8
// channels of one tap; kPair two neighbouring taps of 16-byte pixels (layers of at most four channels).
enum { kPoint, kTaps, kPair };

struct F32Params {
    const char* x;
    const char* wp;
    const float *bias, *residual, *slope, *bn_a, *bn_b;
    float *y, *y_nchw;
    unsigned pixels, x_bytes, w_bytes, items;
    unsigned fast;                 // the channel groups or (tiles_fast) the pixel tiles, whichever neighbouring items walk
    unsigned fast_magic, image_magic, width_magic;  // exhip_divide() by fast, out_h * out_w, out_w
    int fast_shift, image_shift, width_shift, tiles_fast;
    int in_h, in_w, out_h, out_w, stride, pad_t, pad_l, kh, kw;
    int xs_b, row_b;               // bytes per input pixel and input row
    int csteps, n_ksteps;          // steps per tap (kPair: 1) and in all
    int start_r[kMaxSplit + 1], start_q[kMaxSplit + 1], start_c[kMaxSplit + 1], start_s[kMaxSplit + 1];  // where each wave of a tile begins
    int K, kstride, k_end;         // channels from k_end on are not written
    int act, post_relu, bn_relu, post_op, slope_shared, residual_last;
    float alpha, beta;
    int vector_rows;               // output (and shortcut) rows take 16-byte accesses
    int rstride, res_shift;        // the shortcut's channel stride; log2 of how many output pixels per axis share one of its pixels
    int layout, group;             // EXHIP_PLACE_*; grouped: channels per group, shuffled: channels of an upsampled pixel
};

__device__ __forceinline__ v4f load4(__amdgpu_buffer_rsrc_t r, unsigned voff, int soff) {
    return __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(r, (int)voff, soff, 0));
}

// The epilogue of a tile whose blocks four waves or more share: V channels from ch0 on of the lane's pixel. Each wave takes an equal part of
// the tile, so that its chain is short, and stores from registers: a launch that splits its tiles so far is small, and the waves fill the same
// lines. (One wave finished a whole block before, 2400 to 5300 cycles of a launch's 10 000 to 16 000: 512 -> 512 1x1 on three 13 x 13 maps
// 6.9 -> 6.5 us, 256 -> 128 1x1 on three 26 x 26 maps 5.8 -> 5.3.)
constexpr int kParams = 4;                // bias / PReLU slope / BatchNorm a / b

template <int V, bool SLOW = false>
__device__ __forceinline__ void epilogue_part(const F32Params& p, float (&v)[V], const float (&par)[kParams][V], const float (&res)[V], unsigned pix, unsigned img,
                                              unsigned in_image, int ch0) {
    const unsigned per_image = (unsigned)(p.out_h * p.out_w);
    auto relu = [&]() {
#pragma unroll
        for (int e = 0; e < V; ++e) v[e] = (0.f > v[e]) ? 0.f : v[e];
    };
    auto each = [&](auto op) {
#pragma unroll
        for (int e = 0; e < V; ++e) v[e] = unary_value<decltype(op)::value>(v[e], p.alpha, p.beta);
    };
#pragma unroll
    for (int e = 0; e < V; ++e) v[e] += par[0][e];
    if (p.act == 1) relu();
    if (p.act == 3 || SLOW) {
#pragma unroll
        for (int e = 0; e < V; ++e) v[e] = exhip_act(v[e], SLOW ? p.act : 3);
    }
    if (p.residual && !p.residual_last) {
#pragma unroll
        for (int e = 0; e < V; ++e) v[e] += res[e];
    }
    if (p.post_relu) relu();
    if (p.bn_a) {
#pragma unroll
        for (int e = 0; e < V; ++e) v[e] = __builtin_fmaf(par[3][e], v[e], par[2][e]);
        if (p.bn_relu) relu();
    }
    switch (p.post_op) {
    case 0: break;
    case 1 + EXHIP_UNARY_HARDSWISH: each(std::integral_constant<int, 0>{}); break;
    case 1 + EXHIP_UNARY_LEAKYRELU: each(std::integral_constant<int, 1>{}); break;
    case 1 + EXHIP_UNARY_HARDSIGMOID: each(std::integral_constant<int, 3>{}); break;
    case 1 + EXHIP_UNARY_CLIP: each(std::integral_constant<int, 4>{}); break;
    default:
#pragma unroll
        for (int e = 0; e < V; ++e) v[e] = v[e] >= 0.f ? v[e] : par[1][e] * v[e];
    }
    if (p.residual && p.residual_last) {
#pragma unroll
        for (int e = 0; e < V; ++e) v[e] += res[e];
    }
    if (pix >= p.pixels) return;
    if (p.y) {
#pragma unroll
        for (int e = 0; e < V; ++e)
            if (ch0 + e >= p.K) v[e] = 0.f;  // pad channels hold zeros
        if (p.layout == EXHIP_PLACE_GROUPED) {
            // y[img][group][pixel][member]
            float* const to = p.y + (size_t)img * (unsigned)p.K * per_image + (size_t)in_image * (unsigned)p.group;
            int g = ch0 / p.group, member = ch0 - g * p.group;
#pragma unroll
            for (int e = 0; e < V; ++e) {
                if (ch0 + e < p.K) to[(size_t)g * per_image * (unsigned)p.group + member] = v[e];
                if (++member == p.group) member = 0, ++g;
            }
        } else {
            float* to = p.y + (size_t)pix * (unsigned)p.kstride + ch0;
            int end = p.k_end, ch = ch0;
            if (p.layout == EXHIP_PLACE_SHUFFLED && p.vector_rows) {
                // channel pos * group + k of pixel (y, x) is channel k of pixel (2 y + pos / 2, 2 x + pos % 2) of a map twice as large
                const unsigned oy = exhip_divide(in_image, (unsigned)p.out_w, p.width_magic, p.width_shift), ox = in_image - oy * (unsigned)p.out_w;
                const int pos = ch0 / p.group;
                const unsigned at = (img * 2 * (unsigned)p.out_h + 2 * oy + (pos >> 1)) * 2 * (unsigned)p.out_w + 2 * ox + (pos & 1);
                to = p.y + (size_t)at * (unsigned)p.kstride + (ch0 - pos * p.group);
                end = p.K;
            }
            if (p.layout == EXHIP_PLACE_SHUFFLED && !p.vector_rows) {
                const unsigned oy = exhip_divide(in_image, (unsigned)p.out_w, p.width_magic, p.width_shift), ox = in_image - oy * (unsigned)p.out_w;
                const unsigned corner = (img * 2 * (unsigned)p.out_h + 2 * oy) * 2 * (unsigned)p.out_w + 2 * ox;
#pragma unroll
                for (int e = 0; e < V; ++e) {
                    const int pos = (ch0 + e) / p.group, k = ch0 + e - pos * p.group;
                    if (ch0 + e < p.K) p.y[(size_t)(corner + (unsigned)(pos >> 1) * 2 * (unsigned)p.out_w + (pos & 1)) * (unsigned)p.kstride + k] = v[e];
                }
            } else if (p.vector_rows) {
#pragma unroll
                for (int e = 0; e < V; e += 4)
                    if (ch + e < end) *reinterpret_cast<v4f*>(to + e) = v4f{v[e], v[e + 1], v[e + 2], v[e + 3]};
            } else {
#pragma unroll
                for (int e = 0; e < V; ++e)
                    if (ch + e < end) to[e] = v[e];
            }
        }
    }
    if (p.y_nchw) {  // 32 neighbouring pixels of a channel per store instruction and half-wave
        float* const dst = p.y_nchw + ((size_t)img * p.K + ch0) * per_image + in_image;
#pragma unroll
        for (int e = 0; e < V; ++e)
            if (ch0 + e < p.K) dst[(size_t)e * per_image] = v[e];
    }
}

}  // namespace
