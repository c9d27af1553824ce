// bottleneck_kernel: the three layers of a mobile network's block -- pointwise to e channels, depthwise 3x3, pointwise to k channels (with the
// sum behind it) -- as one launch on NHWC halves.
//
// As launches of their own the first layer writes a map of e channels, the largest tensor of the block, for the second to read: 64 -> 128 -> 64
// at 64 x 56 x 56 moves 103 of its 154 MB for that, and on one face's maps of 28 x 28 to 7 x 7 each launch is a chain of a few
// microseconds whatever it computes. Here a group of four or eight waves has a tile of output pixels, makes the e channels of the pixels
// under it (its border twice or more: the products are cheap) and keeps them in LDS:
//   the input's pixels -> LDS | first products -> rounded, activation, rounded -> LDS | depthwise, a thread four channels of strips of PX pixels -> LDS |
//   last products -> rows.
// What bounds it: a wave's chain. Alone on a CU the four phases of 4 x 4 pixels of 64 -> 128 -> 64 take 4000, 3700, 3800 and 2200 cycles, 150 of them
// MFMA; an item's weights are therefore requested during the one before, and the activation is six instructions a pair (both: 47.8 -> 43.2 us
// at 64 x 112 x 112 32 -> 64 -> 64, 48.7 -> 44.8 at 64 x 56 x 56 64 -> 128 -> 64). At those sizes the vector instructions of the depthwise sums and of the two
// epilogues fill the SIMDs, against 13 and 9 us for the block's own bytes at 5.8 TB/s.
// Every value is rounded where the layers by themselves store it, and every sum runs in their order (runs of k-steps where the split form of
// conv_pw.hip would take the layer): the results are theirs, bit for bit.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <mutex>

#include "bottleneck.h"

namespace {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef exhip_v4i v4i;
typedef int v2i __attribute__((ext_vector_type(2)));
typedef short v2s __attribute__((ext_vector_type(2)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));

constexpr unsigned kRsrcWord3 = 0x00020000u;   // raw buffer: out-of-range loads return 0, such stores are dropped
constexpr int kOutOfRange = 0x7ffff000;        // a lane offset beyond every view
constexpr int kRuns = 4;
constexpr int kSlicePitch = 64 + 16;           // a pixel's 32 channels in a wave's slice, and padding
constexpr int kLdsLimit = 160 * 1024;

// A pointwise layer's products: packed weights, k-steps, blocks per packed slab, and where the runs of its sums begin (one run: the end).
struct Products {
    const char* wp;
    const float* bias;
    int w_bytes, steps, mts, channels, start[kRuns + 1], runs;
};

struct BottleneckParams {
    const char* x;
    Products first, last;
    const float* slope;                // PReLU behind the first layer
    const float *dw_w, *dw_bias, *dw_slope;
    const uint16_t* residual;
    uint16_t* y;
    unsigned x_bytes;
    int slope_shared, relu, dw_slope_shared, dw_act;
    int in_h, in_w, out_h, out_w, pad_t, pad_l;
    int pixel_b;                       // bytes per input pixel
    int th, tw, ih, iw;                // a tile's output pixels, and the pixels under it
    exhip_divisor by_tiles, by_tiles_x, by_pieces, by_iw, by_tw, by_strips, by_channels4;
    int tiles, tiles_x, strips_x;      // tiles per image and per row of tiles, strips per row of a tile
    int params_at, wide_at, narrow_at, mid_at;  // LDS: the first layer's parameters; its results; the input's pixels, later depthwise weights and results
};

__device__ __forceinline__ void round_halves(float (&v)[16]) {
#pragma unroll
    for (int e = 0; e < 16; e += 2) {
        const unsigned d = exhip_round_pair(v[e], v[e + 1]);
        v[e] = exhip_h2f((uint16_t)(d & 0xffff));
        v[e + 1] = exhip_h2f((uint16_t)(d >> 16));
    }
}

// PReLU of two values, rounded in front of it and behind it: the product where the sign is set. (A negative zero times a negative slope is a positive
// zero here; the sums behind begin with one, so nothing follows from that.)
// Sixteen bits of a sign by one packed shift and the selection by one v_bfi: left to itself the compiler takes the pair apart (14 instructions for 6).
__device__ __forceinline__ unsigned prelu_pair(float lo, float hi, float slope_lo, float slope_hi) {
    const unsigned h = exhip_round_pair(lo, hi);
    const v2h v = __builtin_bit_cast(v2h, h);
    const unsigned below = exhip_round_pair(__builtin_fmaf((float)v[0], slope_lo, 0.f), __builtin_fmaf((float)v[1], slope_hi, 0.f));
    unsigned negative;
    asm("v_pk_ashrrev_i16 %0, %1, %2" : "=v"(negative) : "v"(0x000f000f), "v"(h));
    return (below & negative) | (h & ~negative);
}

// Products of one 32-channel block with N blocks of 32 pixels in LDS, in runs. a: the first R k-steps, requested before; left with those of the block at
// w_next (where that is not negative), which are on their way while this block's results are finished.
template <bool RUNS, int N, int R>
__device__ __forceinline__ void block_products(const Products& l, __amdgpu_buffer_rsrc_t wr, int w_base, int w_next, int lane, v4i (&a)[R], const char* const (&src)[N],
                                               v16f (&acc)[N]) {
    v16f sum[RUNS ? N : 1];
#pragma unroll
    for (int n = 0; n < N; ++n)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[n][e] = sum[RUNS ? n : 0][e] = 0.f;
    const int w_step = l.mts * 1024;
    int run = 1, end = l.start[1];
    for (int s = 0; s < l.steps; s += R) {
#pragma unroll
        for (int u = 0; u < R; ++u) {
            if (s + u < l.steps) {
                if (RUNS && s + u == end) {
#pragma unroll
                    for (int n = 0; n < N; ++n)
#pragma unroll
                        for (int e = 0; e < 16; ++e) sum[RUNS ? n : 0][e] += acc[n][e], acc[n][e] = 0.f;
                    do end = l.start[++run]; while (end == s + u);
                }
#pragma unroll
                for (int n = 0; n < N; ++n)
                    acc[n] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, a[u]), *reinterpret_cast<const v8h*>(src[n] + (s + u) * 32), acc[n], 0, 0, 0);
                const int at = s + u + R < l.steps ? w_base + (s + u + R) * w_step : w_next < 0 ? -1 : w_next + u * w_step;
                if (at >= 0) a[u] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(wr, lane * 16, at, 0));
            }
        }
    }
    if (RUNS && l.runs > 1) {
#pragma unroll
        for (int n = 0; n < N; ++n)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[n][e] = sum[RUNS ? n : 0][e] + acc[n][e];
    }
}

// RUNS: 0 neither layer's sums in runs, 1 the last one's (the usual case: four waves a SIMD still), 2 both
template <int S, int PX, int WAVES, int RUNS>
__global__ __launch_bounds__(64 * WAVES, RUNS == 2 ? 3 : 4) void bottleneck_kernel(const BottleneckParams p) {
    exhip_touch_args(p);
    constexpr int THREADS = 64 * WAVES, R = 4, NC = (PX - 1) * S + 3, XB = 4;
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), half = lane >> 5;
    unsigned group = blockIdx.x;
    {
        const unsigned per = gridDim.x >> 3;  // one contiguous run of tiles per XCD: neighbours share the pixels of their borders
        if (group < (per << 3)) group = (group & 7) * per + (group >> 3);
    }
    const unsigned img = __builtin_amdgcn_readfirstlane(p.by_tiles(group)), in_image = group - img * (unsigned)p.tiles;
    const unsigned ty = __builtin_amdgcn_readfirstlane(p.by_tiles_x(in_image)), tx = in_image - ty * (unsigned)p.tiles_x;
    const int oy0 = (int)ty * p.th, ox0 = (int)tx * p.tw, iy0 = oy0 * S - p.pad_t, ix0 = ox0 * S - p.pad_l;
    const int wide = p.first.channels, under = p.ih * p.iw, pixels = p.th * p.tw;
    char* const in_lds = lds + p.narrow_at;
    char* const wide_lds = lds + p.wide_at;
    const int in_pitch = p.pixel_b + 16, wide_pitch = wide * 2 + 16;
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(p.x), 0, (int)p.x_bytes, kRsrcWord3);
    const __amdgpu_buffer_rsrc_t wr1 = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(p.first.wp), 0, p.first.w_bytes, kRsrcWord3);
    const __amdgpu_buffer_rsrc_t wr2 = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(p.last.wp), 0, p.last.w_bytes, kRsrcWord3);
    auto weights_at = [](const Products& l, int kb) { return ((kb >> (l.mts >> 1)) * l.steps * l.mts + (kb & (l.mts - 1))) * 1024; };
    v4i a[R];
    auto request = [&](const Products& l, __amdgpu_buffer_rsrc_t wr, int w_base) {
#pragma unroll
        for (int u = 0; u < R; ++u) a[u] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(wr, lane * 16, w_base + (u < l.steps ? u : l.steps - 1) * l.mts * 1024, 0));
    };

    // ---- the input's pixels under the tile ----
    const int pieces = p.pixel_b >> 4;
    request(p.first, wr1, weights_at(p.first, wave % (wide / 32)));
    {
        const int total = under * pieces;
        const unsigned image_at = img * (unsigned)(p.in_h * p.in_w * p.pixel_b);
        for (int base = threadIdx.x; base < total; base += THREADS * XB) {
            v4i r[XB];
            int to[XB];
#pragma unroll
            for (int j = 0; j < XB; ++j) {
                const int i = base + j * THREADS, pixel = (int)p.by_pieces((unsigned)i), piece = i - pixel * pieces;
                const int row = (int)p.by_iw((unsigned)pixel), col = pixel - row * p.iw, iy = iy0 + row, ix = ix0 + col;
                const bool in = i < total && (unsigned)iy < (unsigned)p.in_h && (unsigned)ix < (unsigned)p.in_w;
                to[j] = i < total ? pixel * in_pitch + piece * 16 : -1;
                r[j] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(xr, in ? (int)(image_at + (unsigned)((iy * p.in_w + ix) * p.pixel_b + piece * 16)) : kOutOfRange, 0, 0));
            }
#pragma unroll
            for (int j = 0; j < XB; ++j)
                if (to[j] >= 0) *reinterpret_cast<v4i*>(in_lds + to[j]) = r[j];
        }
        float* const params = reinterpret_cast<float*>(lds + p.params_at);
        for (int c = threadIdx.x; c < wide; c += THREADS) {
            params[c] = p.first.bias ? p.first.bias[c] : 0.f;
            if (p.slope) params[wide + c] = p.slope[p.slope_shared ? 0 : c];
        }
    }
    // what the depthwise layer needs of a thread's four channels: weights (through LDS, once the input's pixels are done with), bias, slopes
    const int channels4 = wide >> 2, weight_pieces = channels4 * 9;
    constexpr int kAhead = 2;
    v4f piece[kAhead];
#pragma unroll
    for (int q = 0; q < kAhead; ++q) piece[q] = reinterpret_cast<const v4f*>(p.dw_w)[min((int)threadIdx.x + q * THREADS, weight_pieces - 1)];
    const int first_strip = (int)p.by_channels4(threadIdx.x), g = (int)threadIdx.x - first_strip * channels4, strip_lanes = (int)p.by_channels4(THREADS);
    float b[4], sl[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        b[e] = p.dw_bias ? p.dw_bias[g * 4 + e] : 0.f;
        sl[e] = p.dw_slope ? p.dw_slope[p.dw_slope_shared ? 0 : g * 4 + e] : 0.f;
    }
    __syncthreads();

    // ---- the first layer: items of a 32-channel block and two blocks of the pixels ----
    {
        const int kblocks = wide >> 5, blocks = (under + 31) >> 5, items = kblocks * ((blocks + 1) >> 1);
        int kb = wave, pair = 0;
        while (kb >= kblocks) kb -= kblocks, ++pair;
        int w_base = weights_at(p.first, kb);
        for (int item = wave; item < items; item += WAVES) {
            int kb_next = kb + WAVES, pair_next = pair;
            while (kb_next >= kblocks) kb_next -= kblocks, ++pair_next;
            const int w_next = weights_at(p.first, kb_next);
            const char* src[2];
            int pixel[2];
            bool in[2];
#pragma unroll
            for (int n = 0; n < 2; ++n) {
                pixel[n] = (pair * 2 + n) * 32 + (lane & 31);
                const int at = pixel[n] < under ? pixel[n] : under - 1;
                src[n] = in_lds + at * in_pitch + half * 16;
                const int row = (int)p.by_iw((unsigned)at), iy = iy0 + row, ix = ix0 + at - row * p.iw;
                in[n] = (unsigned)iy < (unsigned)p.in_h && (unsigned)ix < (unsigned)p.in_w;
            }
            v16f acc[2];
            block_products<RUNS == 2, 2, R>(p.first, wr1, w_base, item + WAVES < items ? w_next : -1, lane, a, src, acc);
            float bias[16], slope[16];
            const float* const params = reinterpret_cast<const float*>(lds + p.params_at) + kb * 32 + half * 16;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const v4f t = *reinterpret_cast<const v4f*>(params + q * 4);
#pragma unroll
                for (int e = 0; e < 4; ++e) bias[q * 4 + e] = t[e];
            }
            if (p.slope) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const v4f t = *reinterpret_cast<const v4f*>(params + wide + q * 4);
#pragma unroll
                    for (int e = 0; e < 4; ++e) slope[q * 4 + e] = t[e];
                }
            }
#pragma unroll
            for (int n = 0; n < 2; ++n) {
                if (pair * 2 + n >= blocks) break;
                float v[16];
#pragma unroll
                for (int e = 0; e < 16; ++e) v[e] = acc[n][e] + bias[e];
                unsigned o[8];
                if (p.slope) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) o[e] = prelu_pair(v[2 * e], v[2 * e + 1], slope[2 * e], slope[2 * e + 1]);
                } else {
                    if (p.relu) {
#pragma unroll
                        for (int e = 0; e < 16; ++e) v[e] = (0.f > v[e]) ? 0.f : v[e];
                    }
#pragma unroll
                    for (int e = 0; e < 8; ++e) o[e] = exhip_round_pair(v[2 * e], v[2 * e + 1]);
                }
#pragma unroll
                for (int e = 0; e < 8; ++e) o[e] = in[n] ? o[e] : 0;  // the depthwise layer's padding
                if (pixel[n] < under) {
                    char* const to = wide_lds + pixel[n] * wide_pitch + kb * 64 + half * 32;
                    *reinterpret_cast<v4i*>(to) = v4i{(int)o[0], (int)o[1], (int)o[2], (int)o[3]};
                    *reinterpret_cast<v4i*>(to + 16) = v4i{(int)o[4], (int)o[5], (int)o[6], (int)o[7]};
                }
            }
            kb = kb_next, pair = pair_next, w_base = w_next;
        }
    }
    __syncthreads();

    // ---- the depthwise layer ----
    v4f* const wk = reinterpret_cast<v4f*>(in_lds);
#pragma unroll
    for (int q = 0; q < kAhead; ++q)
        if ((int)threadIdx.x + q * THREADS < weight_pieces) wk[threadIdx.x + q * THREADS] = piece[q];
    for (int i = threadIdx.x + kAhead * THREADS; i < weight_pieces; i += THREADS) wk[i] = reinterpret_cast<const v4f*>(p.dw_w)[i];
    const int out_blocks = (p.last.channels + 31) >> 5, pixel_blocks = (pixels + 31) >> 5, tiles = out_blocks * pixel_blocks;
    int kb = wave, sub = 0;
    while (kb >= out_blocks) kb -= out_blocks, ++sub;
    int w_base = weights_at(p.last, kb);
    request(p.last, wr2, w_base);  // on their way while the depthwise results are made
    __syncthreads();
    char* const mid = lds + p.mid_at;
    {
        float k[36];
#pragma unroll
        for (int q = 0; q < 9; ++q) {
            const v4f t = wk[g * 9 + q];
#pragma unroll
            for (int e = 0; e < 4; ++e) k[q * 4 + e] = t[e];
        }
        const int strips = first_strip < strip_lanes ? p.th * p.strips_x : 0;
        for (int st = first_strip; st < strips; st += strip_lanes) {
            const int oy = (int)p.by_strips((unsigned)st), ox = (st - oy * p.strips_x) * PX;
            const char* const from = wide_lds + (oy * S * p.iw + ox * S) * wide_pitch + g * 8;
            v4h r[3][NC];
#pragma unroll
            for (int i = 0; i < 3; ++i)
#pragma unroll
                for (int c = 0; c < NC; ++c) r[i][c] = *reinterpret_cast<const v4h*>(from + (i * p.iw + c) * wide_pitch);
#pragma unroll
            for (int px = 0; px < PX; ++px) {
                v4f res;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    float sum = b[e];
#pragma unroll
                    for (int j = 0; j < 3; ++j) {
                        float s = 0.f;
#pragma unroll
                        for (int i = 0; i < 3; ++i) s = __builtin_fmaf((float)r[i][px * S + j][e], k[e * 9 + i * 3 + j], s);
                        sum += s;
                    }
                    res[e] = sum;
                }
                v2i o;
                if (p.dw_slope) {
                    o = v2i{(int)prelu_pair(res[0], res[1], sl[0], sl[1]), (int)prelu_pair(res[2], res[3], sl[2], sl[3])};
                } else {
                    if (p.dw_act != 0) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            res[e] = (0.f > res[e]) ? 0.f : res[e];
                            if (p.dw_act == 3) res[e] = res[e] <= 6.f ? res[e] : 0.f;
                        }
                    }
                    o = v2i{(int)exhip_round_pair(res[0], res[1]), (int)exhip_round_pair(res[2], res[3])};
                }
                *reinterpret_cast<v2i*>(mid + (oy * p.tw + ox + px) * wide_pitch + g * 8) = o;
            }
        }
    }
    __syncthreads();

    // ---- the last layer: 32 channels x 32 pixels at a time ----
    char* const slice = wide_lds + wave * (32 * kSlicePitch);  // (the first layer's results are no longer read)
    for (int item = wave; item < tiles; item += WAVES) {
        int kb_next = kb + WAVES, sub_next = sub;
        while (kb_next >= out_blocks) kb_next -= out_blocks, ++sub_next;
        const int w_next = weights_at(p.last, kb_next);
        const int slot = sub * 32 + (lane & 31), at = slot < pixels ? slot : pixels - 1;
        const int py = (int)p.by_tw((unsigned)at), px = at - py * p.tw, oy = oy0 + py, ox = ox0 + px;
        const bool mine = slot < pixels && oy < p.out_h && ox < p.out_w;
        const size_t row_at = ((size_t)(img * (unsigned)p.out_h + (unsigned)oy) * (unsigned)p.out_w + (unsigned)ox) * (unsigned)p.last.channels;
        const int ch0 = kb * 32 + half * 16;
        v4i res[2] = {};
        if (p.residual && mine && ch0 < p.last.channels) {
            res[0] = *reinterpret_cast<const v4i*>(p.residual + row_at + ch0);
            res[1] = *reinterpret_cast<const v4i*>(p.residual + row_at + ch0 + 8);
        }
        const __amdgpu_buffer_rsrc_t br = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.last.bias), 0, p.last.bias ? p.last.channels * 4 : 0, kRsrcWord3);
        v4f bias[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) bias[q] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(br, (ch0 + q * 4) * 4, 0, 0));
        const char* const src[1] = {mid + at * wide_pitch + half * 16};
        v16f acc[1];
        block_products<RUNS != 0, 1, R>(p.last, wr2, w_base, item + WAVES < tiles ? w_next : -1, lane, a, src, acc);
        float v[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) v[e] = acc[0][e] + bias[e >> 2][e & 3];
        if (p.residual) {
            round_halves(v);
#pragma unroll
            for (int e = 0; e < 16; ++e) v[e] += exhip_h2f((uint16_t)((unsigned)res[e >> 3][(e >> 1) & 3] >> ((e & 1) * 16) & 0xffff));
        }
        v4i o[2];
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e >> 2][e & 3] = (int)exhip_round_pair(v[2 * e], v[2 * e + 1]);
        *reinterpret_cast<v4i*>(slice + (lane & 31) * kSlicePitch + half * 32) = o[0];
        *reinterpret_cast<v4i*>(slice + (lane & 31) * kSlicePitch + half * 32 + 16) = o[1];
        // four neighbouring lanes store a pixel's 64 bytes
        const unsigned place = mine ? (unsigned)(oy * p.out_w + ox) : 0xffffffffu;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int row = j * 16 + (lane >> 2), col = (lane & 3) * 8;
            const unsigned to = (unsigned)__builtin_amdgcn_ds_bpermute(row * 4, (int)place);
            if (to != 0xffffffffu && kb * 32 + col < p.last.channels)
                *reinterpret_cast<v4i*>(p.y + ((size_t)img * (unsigned)(p.out_h * p.out_w) + to) * (unsigned)p.last.channels + kb * 32 + col) =
                    *reinterpret_cast<const v4i*>(slice + row * kSlicePitch + col * 2);
        }
        kb = kb_next, sub = sub_next, w_base = w_next;
    }
}

std::mutex g_attr_mutex;

template <int S, int PX, int WAVES, int RUNS>
int go(exhip_ctx* ctx, const BottleneckParams& p, unsigned groups, int lds) {
    auto kernel = bottleneck_kernel<S, PX, WAVES, RUNS>;
    {
        static unsigned long long attr_set = 0;
        std::lock_guard<std::mutex> lock(g_attr_mutex);
        const unsigned long long bit = 1ull << (ctx->device & 63);
        if (!(attr_set & bit)) {
            EXHIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kLdsLimit));
            attr_set |= bit;
        }
    }
    hipLaunchKernelGGL(kernel, dim3(groups), dim3(64 * WAVES), lds, ctx->stream, p);
    EXHIP_LAUNCH_CHECK();
    return 0;
}

template <int WAVES, int RUNS>
int pick(exhip_ctx* ctx, const BottleneckParams& p, int stride, int px, unsigned groups, int lds) {
    if (stride == 2) return px == 2 ? go<2, 2, WAVES, RUNS>(ctx, p, groups, lds) : go<2, 1, WAVES, RUNS>(ctx, p, groups, lds);
    return px == 4 ? go<1, 4, WAVES, RUNS>(ctx, p, groups, lds) : px == 2 ? go<1, 2, WAVES, RUNS>(ctx, p, groups, lds) : go<1, 1, WAVES, RUNS>(ctx, p, groups, lds);
}

Products products(const exhip_bottleneck_layer& l) {
    Products q = {};
    q.wp = static_cast<const char*>(l.wp);
    q.bias = l.bias;
    q.w_bytes = (int)l.w_bytes;
    q.steps = l.steps;
    q.mts = l.slab_blocks;
    q.channels = l.channels;
    q.runs = l.runs;
    for (int i = 0; i <= kRuns; ++i) q.start[i] = i == 0 ? 0 : i < l.runs ? l.start[i] : l.steps;
    return q;
}

int strip_pixels(int tw, int stride) { return tw % 4 == 0 && stride == 1 ? 4 : tw % 2 == 0 ? 2 : 1; }  // (four at stride 2 spill)

struct Areas {  // of the LDS
    int wide_at, narrow_at, mid_at, end;
    Areas(const exhip_bottleneck& b, int th, int tw, int waves) {
        const int wide = b.first.channels, pitch = wide * 2 + 16, under = ((th - 1) * b.stride + 3) * ((tw - 1) * b.stride + 3);
        wide_at = (b.slope ? 2 : 1) * wide * 4;
        narrow_at = wide_at + std::max(under * pitch, waves * 32 * kSlicePitch);
        mid_at = narrow_at + wide * 36;
        end = narrow_at + std::max(under * (b.pixel_b + 16), wide * 36 + th * tw * pitch);
    }
};

struct Plan {
    int th = 0, tw = 0, waves = 0;  // waves 0: the layers by themselves
};

// The tile and the waves by a model of the launch, in microseconds: 3.0 for the launch; per round of groups 0.24, 0.56 for each pass over the
// threads that stages the input, 0.53 and 0.113 per k-step for a wave's item of the first products, 0.6 and 0.073 for one of the last ones, 0.115
// and 0.27 per pixel for a thread's strip; a wave of a SIMD's w takes 1 + 0.22 (w - 1) times as long as one alone, and never less than 0.3 w. Fitted to 45
// blocks (1 to 64 maps of 7 x 7 to 160 x 160, 16 to 1024 channels) in 30 to 50 tiles each, it picks one 2 % slower than the fastest on
// average. The layers by themselves are a launch each, or two, their maps at 6.8 TB/s, their products at 0.4 PFLOP/s and 0.065 for
// every k-step of the two chains: where that is shorter they stay (1 x 14 x 14 128 -> 512 -> 128 10.6 us against 11.9, 64 x 7 x 7
// 512 -> 1024 -> 512 33.5 against 39.3: a group's chain through all channels is too long); of the 45 none went the wrong way. us, the layers ->
// the block: 64 x 112 x 112 32 -> 64 -> 64 at stride 2 58.2 -> 43.3, 64 x 56 x 56 64 -> 128 -> 64 56.3 -> 44.5, 64 x 28 x 28 128 -> 256 -> 128
// 39.6 -> 31.5, 64 x 14 x 14 256 -> 512 -> 256 37.0 -> 29.0, 16 x 56 x 56 64 -> 128 -> 64 20.9 -> 14.9, 1 x 28 x 28 8.4 -> 6.4.
Plan choose(const exhip_bottleneck& b) {
    static const unsigned char kTiles[][2] = {{1, 4}, {1, 7}, {2, 2}, {2, 4}, {2, 5}, {4, 2}, {3, 4}, {2, 7}, {8, 2}, {4, 4}, {4, 5}, {5, 5}, {6, 4}, {7, 4}, {4, 7}, {4, 8}, {6, 8}, {7, 7}, {8, 8}, {4, 14}, {8, 14}};
    const int wide = b.first.channels, k = b.last.channels, out_blocks = (k + 31) / 32;
    const double in_px = (double)b.n * b.in_h * b.in_w, out_px = (double)b.n * b.out_h * b.out_w;
    double best = 7.3 + (in_px * (b.pixel_b + 4 * wide) + out_px * k * 2) / 6.8e6 + (in_px * (b.pixel_b / 2) + out_px * k) * wide * 5.1e-9 + 0.065 * (b.first.steps + b.last.steps);
    Plan plan;
    for (const auto& t : kTiles) {
        const int th = t[0], tw = t[1], under = ((th - 1) * b.stride + 3) * ((tw - 1) * b.stride + 3);
        if (th > b.out_h + 1 || tw > b.out_w + 3 || (b.stride == 2 && th * tw > 64)) continue;
        const long long groups = (long long)b.n * ((b.out_h + th - 1) / th) * ((b.out_w + tw - 1) / tw);
        const int px = strip_pixels(tw, b.stride), pairs = ((under + 31) / 32 + 1) / 2;
        for (int waves = 4; waves <= 8; waves += 4) {
            const int lds = (Areas(b, th, tw, waves).end + 1279) / 1280 * 1280;
            if (lds > kLdsLimit) continue;
            const int resident = std::max(1, std::min(kLdsLimit / lds, (b.first.runs > 1 ? 12 : 16) / waves)), lanes = std::max(1, 64 * waves / (wide / 4));
            auto times = [&](int n) { return (double)((n + waves - 1) / waves); };
            const double chain = 0.24 + 0.56 * ((under * (b.pixel_b / 16) + 256 * waves - 1) / (256 * waves)) + times(wide / 32 * pairs) * (0.53 + 0.113 * b.first.steps) +
                                 (th * (tw / px) + lanes - 1) / lanes * (0.115 + 0.27 * px) + times(out_blocks * ((th * tw + 31) / 32)) * (0.6 + 0.073 * b.last.steps);
            auto round = [&](long long n) {
                const double w = (double)((n + 255) / 256) * waves / 4;
                return n ? chain * std::max(1 + 0.22 * std::max(w - 1, 0.), (waves == 4 ? 0.3 : 0.315) * w) : 0.;
            };
            const long long slots = 256ll * resident, full = groups / slots;
            const double time = 3.0 + full * round(slots) + round(groups - full * slots);
            if (time < best) {
                best = time;
                plan.th = th; plan.tw = tw; plan.waves = waves;
            }
        }
    }
    return plan;
}

// A thread keeps the plans of its last blocks: the search takes a few microseconds.
Plan plan_of(const exhip_bottleneck& b, int option) {
    if (option > 1) {
        Plan plan;
        plan.th = std::max(1, option / 16 % 16); plan.tw = std::max(1, option % 16); plan.waves = option >= 256 ? 8 : 4;
        return plan;
    }
    const int key[] = {b.n, b.in_h, b.in_w, b.out_h, b.out_w, b.stride, b.pixel_b, b.first.channels, b.last.channels, b.first.runs, b.slope != nullptr};
    constexpr int kKey = sizeof(key) / sizeof(key[0]);
    struct Entry {
        int key[kKey];
        Plan plan;
    };
    static thread_local Entry cache[32] = {};
    Entry& e = cache[(unsigned)(b.n * 13 + b.in_h * 7 + b.in_w * 5 + b.pixel_b / 32 * 3 + b.first.channels / 32 * 11 + b.last.channels / 16 + b.stride) % 32];
    if (!std::equal(key, key + kKey, e.key)) {
        e.plan = choose(b);
        std::copy(key, key + kKey, e.key);
    }
    return e.plan;
}

}  // namespace

int exhip_bottleneck_run(exhip_ctx* ctx, const exhip_bottleneck& b) {
    const int option = g_exhip_options.bottleneck, wide = b.first.channels, k = b.last.channels;
    if (option == 0 || wide % 32 != 0 || wide > 1024 || k % 16 != 0 || k > 1024 || b.pixel_b % 32 != 0 || b.pixel_b > 1024 || (b.stride != 1 && b.stride != 2) ||
        (b.dw_act != 0 && b.dw_act != 1 && b.dw_act != 3) || b.first.w_bytes >= kOutOfRange || b.last.w_bytes >= kOutOfRange ||
        (long long)b.n * b.in_h * b.in_w * b.pixel_b >= (1ll << 30) || (long long)b.out_h * b.out_w >= (1ll << 30))
        return EXHIP_ERR_UNSUPPORTED;
    BottleneckParams p = {};
    p.x = static_cast<const char*>(b.x);
    p.first = products(b.first);
    p.last = products(b.last);
    p.slope = b.slope; p.slope_shared = b.slope_shared; p.relu = b.relu;
    p.dw_w = b.dw_w; p.dw_bias = b.dw_bias; p.dw_slope = b.dw_slope; p.dw_slope_shared = b.dw_slope_shared; p.dw_act = b.dw_act;
    p.residual = b.residual;
    p.y = b.y;
    p.x_bytes = (unsigned)((long long)b.n * b.in_h * b.in_w * b.pixel_b);
    p.in_h = b.in_h; p.in_w = b.in_w; p.out_h = b.out_h; p.out_w = b.out_w; p.pad_t = b.pad_t; p.pad_l = b.pad_l;
    p.pixel_b = b.pixel_b;
    const Plan plan = plan_of(b, option);
    const int waves = plan.waves;
    if (!waves) return EXHIP_ERR_UNSUPPORTED;
    p.th = plan.th;
    p.tw = plan.tw;
    const int px = strip_pixels(p.tw, b.stride);
    p.ih = (p.th - 1) * b.stride + 3;
    p.iw = (p.tw - 1) * b.stride + 3;
    p.strips_x = p.tw / px;
    p.tiles_x = (b.out_w + p.tw - 1) / p.tw;
    p.tiles = p.tiles_x * ((b.out_h + p.th - 1) / p.th);
    p.by_tiles.set((unsigned)p.tiles); p.by_tiles_x.set((unsigned)p.tiles_x); p.by_pieces.set((unsigned)(b.pixel_b / 16)); p.by_iw.set((unsigned)p.iw);
    p.by_tw.set((unsigned)p.tw); p.by_strips.set((unsigned)p.strips_x); p.by_channels4.set((unsigned)(wide / 4));
    const Areas areas(b, p.th, p.tw, waves);
    p.params_at = 0;
    p.wide_at = areas.wide_at;
    p.narrow_at = areas.narrow_at;
    p.mid_at = areas.mid_at;
    const int lds = areas.end;
    const long long groups = (long long)b.n * p.tiles;
    if (lds > kLdsLimit || groups >= (1ll << 30)) return EXHIP_ERR_UNSUPPORTED;
    const int runs = p.first.runs > 1 ? 2 : p.last.runs > 1 ? 1 : 0;
    if (waves == 8)
        return runs == 2 ? pick<8, 2>(ctx, p, b.stride, px, (unsigned)groups, lds) : runs ? pick<8, 1>(ctx, p, b.stride, px, (unsigned)groups, lds) : pick<8, 0>(ctx, p, b.stride, px, (unsigned)groups, lds);
    return runs == 2 ? pick<4, 2>(ctx, p, b.stride, px, (unsigned)groups, lds) : runs ? pick<4, 1>(ctx, p, b.stride, px, (unsigned)groups, lds) : pick<4, 0>(ctx, p, b.stride, px, (unsigned)groups, lds);
}
