// conv3x3_thirds_kernel: float32 convolution with 3x3 filters of whole 16-channel steps at stride 1 on the bfloat16 matrix units.
//
// float32 products run at a sixteenth of the bfloat16 rate (157 against 2500 TFLOP/s), and a float32 is exactly the sum of three bfloat16
// values, its thirds: h = round(x), m = round(x - h), l = x - h - m. Eight of the nine products of two numbers' thirds are taken (all but l l,
// 2^-34 of the result), so that a step of 16 channels costs eight v_mfma_f32_32x32x16_bf16 (256 cycles) instead of eight
// v_mfma_f32_32x32x2_f32 (512). m l and l m, 2^-25 each, are nothing to the sum of many products, whose rounding is larger; a sum of one would be off by up
// to .95 ulp without them. The unit adds 16 products at a
// time and rounds once; it rounds small addends toward minus infinity, though, so h h has accumulators of its own, and the seven
// others, 2^-8 of it, theirs. Against sums in 64 bits the results are off by a third to a half of what the float32 products leave
// (2-norm over K = 576 random values 1.4e-7 and 4.3e-7, over 4608 4.2e-7 and 12.2e-7, all positive 1.3e-7 and 3.7e-7), where only some of the weights are not
// zero by as much for one product, .60 to .98 of it for four.
//
// The weights are packed as thirds. The pixels are split once, on their way into LDS: a group of four or eight waves stages the input
// under a run of pixels, 16 * CS channels at a time, and takes the nine taps from there; a split in registers would cost every wave 44
// vector instructions per 32 pixels, tap and step. Weight fragments come straight from memory, three taps ahead.
//
// A group's pixels are neighbours in a list of the output's vertical strips, row by row (strips.h; a strip of a 13 x 13 map is the map). WK waves share a run's
// steps, their sums meet in LDS in a fixed order.
//
// Bounded by the matrix unit on large maps (128 -> 128 at 16 x 80 x 80 185 us, 164 TFLOP/s of float32 work, conv_f32_kernel 226) and by a group's chain of
// loads, split and products on small ones: us, conv_f32_kernel and this one, launches queued from Python, 64 -> 64 on one 56 x 56 map 6.7, 5.4, at 160 x 160 23.4, 18.8,
// 128 -> 128 at 80 x 80 22.5, 17.8, 512 -> 512 at 20 x 20 24.9, 19.1. Over 62 layers 1.13 times as fast on average, 1.58 at most (112 -> 16 at 22 x 78 x 76), and
// slower where there is little to split for: maps of one pixel .79 to .85, 16 channels in a few groups .81 to .87, 32 and 80 channels there .92 to .99.
//
// What thirds do not hold: a third of an infinity is NaN, as is one times the zero third of a finite weight; below 2^-103 a last third is no normal number, below
// 2^-110 it is cut off, and products below 2^-112 lose their smaller parts. A group that stages a value or finds a sum of that kind computes its
// tile again with float32 products (float32_sums), whose results it gets, all of them; a weight of that kind is packed as a NaN that calls for them (split_weight).
// Such a group takes 2.5 to 3.5 times as long (512 -> 512 at 20 x 20 all NaN 64 us, 128 -> 128 at 4 x 80 x 80 54 -> 184 to 199).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <mutex>

#include "conv_f32.h"
#include "conv_f32_epilogue.h"
#include "strips.h"

namespace {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef unsigned v2u __attribute__((ext_vector_type(2)));

constexpr int kTapBytes = 3 * 1024;          // a 32-channel block's weights of one tap and step: three thirds
constexpr int kStepBytes = 9 * kTapBytes;
constexpr int kLdsLimit = 160 * 1024;

struct ThirdsParams {
    F32Params f;
    exhip_strip_list list;
    exhip_divisor by_fast;
    int chunks;                    // 16 * CS channels each
    int table_b, buffer_b;         // bytes of the tables in front of the staged pixels, and of a buffer of those
    float floor, post_floor;       // `plain`: what the activation and the ReLU behind the shortcut cut off at, -inf: nothing
    int in_place;                  // the results take the shortcut's place
    int plain;                     // results are rows that take 16-byte accesses, and nothing but ReLUs and a shortcut lie behind the products
};

// Two values' thirds, as pairs of bfloat16.
__device__ __forceinline__ unsigned bf16_pair(float a, float b) { return __builtin_bit_cast(unsigned, __builtin_convertvector(v2f{a, b}, v2bf)); }
__device__ __forceinline__ void split_thirds(v4f x, v2u& h, v2u& m, v2u& l) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        float a = x[2 * i], b = x[2 * i + 1];
        h[i] = bf16_pair(a, b);
        a -= __uint_as_float(h[i] << 16);
        b -= __uint_as_float(h[i] & 0xffff0000u);
        m[i] = bf16_pair(a, b);
        a -= __uint_as_float(m[i] << 16);
        b -= __uint_as_float(m[i] & 0xffff0000u);
        l[i] = bf16_pair(a, b);
    }
}

constexpr unsigned kLeast = 0x0c000000;  // 2^-103: every third of a larger float32 is a normal number
constexpr int kNoSum = 0x297;  // v_cmp_class: NaN, infinite or below 2^-126 (and not zero)
__device__ __forceinline__ bool no_sum(float v) { return __builtin_amdgcn_classf(v * 0x1p-14f, kNoSum); }  // nor below 2^-112
constexpr unsigned kWhole = 0x7fff;  // the first third of a weight that thirds do not hold; the others are the halves of its bits

// A weight from its thirds, the even or the odd one of two words of pairs.
__device__ __forceinline__ float whole_weight(unsigned h, unsigned m, unsigned l, bool odd) {
    const unsigned top = odd ? h & 0xffff0000u : h << 16, mid = odd ? m & 0xffff0000u : m << 16, low = odd ? l & 0xffff0000u : l << 16;
    const float sum = __uint_as_float(top) + (__uint_as_float(mid) + __uint_as_float(low));
    return top == kWhole << 16 ? __uint_as_float(mid | low >> 16) : sum;
}

// A wave's sums of the taps [first, last) of all 9 * csteps with float32 products, straight from memory: pix, the lane's pixels in the output. Steps of eight
// v_mfma_f32_32x32x2_f32, the next two taps' operands on their way under a tap's products.
template <int MT, int NT>
__device__ __forceinline__ void float32_sums(const F32Params& p, __amdgpu_buffer_rsrc_t xr, __amdgpu_buffer_rsrc_t wr, int kb0, int first, int last, const unsigned (&pix)[NT], int lane,
                                             v16f (&acc)[MT][NT]) {
    constexpr int R = 2;
    const unsigned per_image = (unsigned)(p.out_h * p.out_w);
    unsigned corner[NT], inside[NT];  // the pixel's top-left input pixel (32-bit wrap-around where it lies in front of the tensor), and which of its taps lie in the image
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        const bool in = pix[n] < p.pixels;
        const unsigned img = exhip_divide(in ? pix[n] : 0, per_image, p.image_magic, p.image_shift), rem = in ? pix[n] - img * per_image : 0;
        const int oy = (int)exhip_divide(rem, (unsigned)p.out_w, p.width_magic, p.width_shift), iy = oy - p.pad_t, ix = (int)rem - oy * p.out_w - p.pad_l;
        corner[n] = (unsigned)((((int)img * p.in_h + iy) * p.in_w + ix) * p.xs_b + (lane >> 5) * 32);
        inside[n] = 0;
#pragma unroll
        for (int tap = 0; tap < 9; ++tap)
            inside[n] |= in && (unsigned)(iy + tap / 3) < (unsigned)p.in_h && (unsigned)(ix + tap % 3) < (unsigned)p.in_w ? 1u << tap : 0u;
    }
    unsigned woff[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) woff[m] = (kb0 + m) * 32 < p.K ? (unsigned)(m * p.csteps * kStepBytes + lane * 16) : kOutOfRange;
    const int w_base = kb0 * p.csteps * kStepBytes;
    v4u a[R][MT][3];
    v4f b[R][NT][2];
    auto request = [&](int u, int at) {  // always: behind a branch the products would wait for all that is on its way. Past the last tap zeros.
        const bool on = at < last;
        const int t = on ? at : last - 1, step = t / 9, tap = t - step * 9, off = tap / 3 * p.row_b + tap % 3 * p.xs_b;
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int i = 0; i < 3; ++i) a[u][m][i] = __builtin_bit_cast(v4u, load4(wr, on ? woff[m] : kOutOfRange, w_base + t * kTapBytes + i * 1024));
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            const unsigned from = on && (inside[n] >> tap & 1) ? corner[n] + (unsigned)off : kOutOfRange;
            b[u][n][0] = load4(xr, from, step * 64);
            b[u][n][1] = load4(xr, from + 16, step * 64);
        }
    };
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[m][n][e] = 0.f;
    if (first >= last) return;
#pragma unroll
    for (int u = 0; u < R; ++u) request(u, first + u);
#pragma unroll 1
    for (int t = first; t < last; t += R) {
#pragma unroll
        for (int u = 0; u < R; ++u) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
#pragma unroll
                for (int m = 0; m < MT; ++m) {
                    const float w = whole_weight(a[u][m][0][i / 2], a[u][m][1][i / 2], a[u][m][2][i / 2], i % 2 != 0);
#pragma unroll
                    for (int n = 0; n < NT; ++n) acc[m][n] = __builtin_amdgcn_mfma_f32_32x32x2f32(w, b[u][n][i / 4][i % 4], acc[m][n], 0, 0, 0);
                }
            }
            request(u, t + u + R);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

// A channel's parameters, zeros for an absent array and beyond the channels.
__device__ __forceinline__ void load_parameters(const F32Params& p, int ch, float (&par)[kParams]) {
    const float* const from[kParams] = {p.bias, p.slope, p.bn_a, p.bn_b};
#pragma unroll
    for (int i = 0; i < kParams; ++i) {
        par[i] = 0.f;
        if (from[i]) {
            const bool shared = i == 1 && p.slope_shared;
            const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(from[i]), 0, shared ? 4 : p.K * 4, kRsrcWord3);
            par[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, shared ? 0 : ch * 4, 0, 0));
        }
    }
}

// How a tile is finished. The waves' sums meet where the pixels were staged, [part][block][four channels][pixel]; a thread finishes four channels of one pixel
// at a time. Eight neighbouring lanes have a pixel's 32 channels, whose 128 bytes they store together, or for a planar result 32
// neighbouring lanes the pixels of a channel. Pixels are dealt out by their channels' number, so that neither side meets bank conflicts.
template <int MT, int NT, int WK>
struct Tail {
    static constexpr int BLOCKS = MT * NT, UNITS = BLOCKS * 4 >= WK ? BLOCKS * 4 / WK : 1;
    static __device__ __forceinline__ bool owner(int part) { return BLOCKS * 4 >= WK || part < BLOCKS * 4; }
    static __device__ __forceinline__ void place(bool planar, int part, int lane, int u, int& block, int& quad, int& row) {
        const int at = (part * 64 + lane + u * WK * 64) % (BLOCKS * 256);
        quad = planar ? at >> 5 & 7 : at & 7;
        row = planar ? at & 31 : at >> 3 & 31;
        block = at >> 8;
    }
};
template <int MT, int NT, int WK>
__device__ __forceinline__ void load_shortcut(const F32Params& p, const unsigned* pixels, int kb0, int part, int side, int lane, v4f (&res)[Tail<MT, NT, WK>::UNITS]) {
    constexpr int UNITS = Tail<MT, NT, WK>::UNITS;
#pragma unroll
    for (int u = 0; u < UNITS; ++u) res[u] = v4f{0.f, 0.f, 0.f, 0.f};
    if (p.residual) {
#pragma unroll
        for (int u = 0; u < UNITS; ++u) {
            int block, quad, row;
            Tail<MT, NT, WK>::place(p.y_nchw != nullptr, part, lane, u, block, quad, row);
            const int ch = (kb0 + block % MT) * 32 + quad * 4;
            unsigned from = pixels[(side * NT + block / MT) * 32 + row];
            if (from >= p.pixels || ch >= p.K) continue;
            if (p.res_shift) {
                const unsigned per_image = (unsigned)(p.out_h * p.out_w), img = exhip_divide(from, per_image, p.image_magic, p.image_shift);
                const unsigned in_image = from - img * per_image, oy = exhip_divide(in_image, (unsigned)p.out_w, p.width_magic, p.width_shift);
                from = (img * ((unsigned)p.out_h >> p.res_shift) + (oy >> p.res_shift)) * ((unsigned)p.out_w >> p.res_shift) +
                       ((in_image - oy * (unsigned)p.out_w) >> p.res_shift);
            }
            const float* const src = p.residual + (size_t)from * (unsigned)p.rstride + ch;
            if (p.vector_rows) {
                res[u] = *reinterpret_cast<const v4f*>(src);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) res[u][e] = ch + e < p.K ? src[e] : 0.f;
            }
        }
    }
}
template <int MT, int NT>
__device__ __forceinline__ void put_sums(const v16f (&acc)[MT][NT], char* red, int part, int lane) {
    constexpr int BLOCKS = MT * NT;
#pragma unroll
    for (int i = 0; i < 4 * BLOCKS; ++i) {
        const v16f& c = acc[i / 4 % MT][i / 4 / MT];
        const int quad = (lane >> 5) * 4 + i % 4;
        *reinterpret_cast<v4f*>(red + part * BLOCKS * 4096 + (i / 4 * 8 + quad) * 512 + ((lane & 31) ^ quad) * 16) =
            v4f{c[i % 4 * 4], c[i % 4 * 4 + 1], c[i % 4 * 4 + 2], c[i % 4 * 4 + 3]};
    }
}
// (whether one of the sums is of a kind that thirds do not hold)
template <int MT, int NT, int WK, bool SLOW>
__device__ __forceinline__ bool finish_tile(const ThirdsParams& q, const unsigned* pixels, const float* params, const char* red, int kb0, int part, int side, int lane,
                                            const v4f (&res)[Tail<MT, NT, WK>::UNITS]) {
    const F32Params& p = q.f;
    constexpr int BLOCKS = MT * NT, UNITS = Tail<MT, NT, WK>::UNITS;
    bool missing = false;
#pragma unroll 1
    for (int u = 0; u < UNITS; ++u) {
        struct {
            unsigned pix;
            int block, quad, row;
            v4f res;
        } now;
        Tail<MT, NT, WK>::place(p.y_nchw != nullptr, part, lane, u, now.block, now.quad, now.row);
        now.pix = pixels[(side * NT + now.block / MT) * 32 + now.row];
        now.res = res[0];
        if (p.residual) {
#pragma unroll
            for (int i = 1; i < UNITS; ++i) now.res = u == i ? res[i] : now.res;
        }
        const char* const from = red + (now.block * 8 + now.quad) * 512 + (now.row ^ now.quad) * 16;
        const float* const my_params = params + now.block % MT * 32 + now.quad * 4;
        const int ch = (kb0 + now.block % MT) * 32 + now.quad * 4;
        v4f sum = *reinterpret_cast<const v4f*>(from);
#pragma unroll
        for (int w = 1; w < WK; ++w) sum += *reinterpret_cast<const v4f*>(from + w * BLOCKS * 4096);
#pragma unroll
        for (int e = 0; e < 4; ++e) missing |= no_sum(sum[e]);
        if (q.plain) {
            const v4f bias = *reinterpret_cast<const v4f*>(my_params);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float v = sum[e] + bias[e];
                v = q.floor > v ? q.floor : v;
                if (p.residual) v += now.res[e];
                v = q.post_floor > v ? q.post_floor : v;
                sum[e] = ch + e < p.K ? v : 0.f;  // pad channels hold zeros
            }
            if (now.pix < p.pixels && ch < p.k_end) *reinterpret_cast<v4f*>(p.y + (size_t)now.pix * (unsigned)p.kstride + ch) = sum;
        } else {
            float v[4], par[kParams][4], res[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[e] = sum[e];
                res[e] = now.res[e];
#pragma unroll
                for (int i = 0; i < kParams; ++i) par[i][e] = my_params[i * MT * 32 + e];
            }
            const unsigned per_image = (unsigned)(p.out_h * p.out_w);
            unsigned img = 0, in_image = 0;
            if (p.y_nchw || p.layout != EXHIP_PLACE_ROWS) {
                img = exhip_divide(now.pix, per_image, p.image_magic, p.image_shift);
                in_image = now.pix - img * per_image;
            }
            epilogue_part<4, SLOW>(p, v, par, res, now.pix, img, in_image, ch);
        }
    }
    return missing;
}

// A tile's results with float32 products, for one that thirds did not do for. A call, so that none of it stands in the way of the others (inlined, scalar registers
// spilled: .1 to .5 us of a small launch). args: where the kernel's arguments are (by reference the parameter would be copied to scratch first).
template <int MT, int NT, int WK, bool SLOW>
__device__ __noinline__ void again_with_floats(const ThirdsParams* args, const unsigned* pixels, const float* params, char* red, int kb0, int part, int side, int lane) {
    const F32Params& p = args->f;
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(p.x), 0, (int)p.x_bytes, kRsrcWord3);
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(p.wp), 0, (int)p.w_bytes, kRsrcWord3);
    unsigned pix[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) pix[n] = pixels[(side * NT + n) * 32 + (lane & 31)];
    v16f acc[MT][NT];
    float32_sums<MT, NT>(p, xr, wr, kb0, 9 * p.csteps * part / WK, 9 * p.csteps * (part + 1) / WK, pix, lane, acc);
    v4f res[Tail<MT, NT, WK>::UNITS];
    load_shortcut<MT, NT, WK>(p, pixels, kb0, part, side, lane, res);
    put_sums<MT, NT>(acc, red, part, lane);
#pragma unroll
    for (int u = 0; u < Tail<MT, NT, WK>::UNITS; ++u) asm volatile("" : "+v"(res[u]));
    __syncthreads();
    if (Tail<MT, NT, WK>::owner(part)) finish_tile<MT, NT, WK, SLOW>(*args, pixels, params, red, kb0, part, side, lane, res);
}

// A wave's tile is 32 * MT channels x 32 * NT pixels; WP waves side by side make a group's run of pixels, WK share the steps of 16 channels,
// of which CS are staged at a time.
template <int MT, int NT, int WK, int WP, int CS, int OCC, bool SLOW>
__global__ __launch_bounds__(64 * WK * WP, OCC) void conv3x3_thirds_kernel(const ThirdsParams q) {
    exhip_touch_args(q);
    const F32Params& p = q.f;
    constexpr int WAVES = WK * WP, THREADS = 64 * WAVES, BLOCKS = MT * NT, RUN = 32 * NT * WP;
    constexpr int PIECES = CS * 4, PASS = THREADS / PIECES;       // 16-byte pieces of a staged pixel; pixels that a pass of the group stages
    constexpr int PITCH = CS * 96 + 16;                           // bytes of a staged pixel: [step][third][16 channels], an odd number of 16s
    constexpr int BATCH = (RUN * 7 / 4 * WK / CS + PASS - 1) / PASS;  // passes whose pixels are on the way at a time
    constexpr int PER_TAP = (BATCH + 5) / 6;                      // of them are put in place under the products of a tap
    static_assert(CS % WK == 0, "every wave has its steps of a chunk");
    extern __shared__ __attribute__((aligned(16))) char lds_all[];
    unsigned* const pixels = reinterpret_cast<unsigned*>(lds_all);   // the run's pixels in the output
    float* const params = reinterpret_cast<float*>(pixels + RUN);    // kParams of the tile's channels
    unsigned* const again = pixels + RUN + kParams * MT * 32;        // whether the tile is computed again
    unsigned* const table = again + 4;                               // where the staged pixels lie in the input
    char* const stage = lds_all + q.table_b;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), half = lane >> 5;
    const int part = wave % WK, side = wave / WK;
    unsigned bid = blockIdx.x;
    {
        const unsigned per = gridDim.x >> 3;  // one contiguous run of items per XCD (conv_f32_kernel)
        if (bid < (per << 3)) bid = (bid & 7) * per + (bid >> 3);
    }
    const unsigned slow = q.by_fast(bid), fast = bid - slow * p.fast;
    const unsigned tile = __builtin_amdgcn_readfirstlane(p.tiles_fast ? fast : slow);
    const int kb0 = __builtin_amdgcn_readfirstlane((int)(p.tiles_fast ? slow : fast) * MT);

    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(p.x), 0, (int)p.x_bytes, kRsrcWord3);
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(p.wp), 0, (int)p.w_bytes, kRsrcWord3);

    // weights: the wave's steps part, part + WK ..., nine taps each
    unsigned woff[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) woff[m] = (kb0 + m) * 32 < p.K && part < p.csteps ? (unsigned)(m * p.csteps * kStepBytes + lane * 16) : kOutOfRange;
    v8bf a[3][MT][3];
    int w_at = (kb0 * p.csteps + part) * kStepBytes;
    auto request = [&](int u, int at) {
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int t = 0; t < 3; ++t) a[u][m][t] = __builtin_bit_cast(v8bf, load4(wr, woff[m], at + t * 1024));
    };

    // the staged rows: those under the run's first pixel to those under its last
    const unsigned run0 = tile * RUN;
    const int first_row = __builtin_amdgcn_readfirstlane(q.list.where<1>(run0, p.out_h, p.out_w).row);
    const int last_row = __builtin_amdgcn_readfirstlane(q.list.where<1>(run0 + RUN - 1, p.out_h, p.out_w).row) + 2;
    const int staged = (last_row - first_row + 1) * q.list.staged_cols;
    if (threadIdx.x == 0) *again = 0;
    for (int i = threadIdx.x; i < staged; i += THREADS) table[i] = q.list.staged_pixel<1>(i, first_row, p.in_h, p.in_w, p.pad_t, p.pad_l, p.xs_b, kOutOfRange);
    __syncthreads();
    v4f x[BATCH];
    const int my_piece = threadIdx.x % PIECES, my_pixel = threadIdx.x / PIECES;
    auto load_batch = [&](int first, int chunk) {
        const int end = chunk * CS * 64 + my_piece * 16 < p.csteps * 64 ? staged : 0;  // (the last chunk may reach beyond the channels)
#pragma unroll
        for (int i = 0; i < BATCH; ++i) {
            const int at = first + i * PASS + my_pixel;
            x[i] = load4(xr, at < end ? table[at] + my_piece * 16 : kOutOfRange, chunk * CS * 64);
        }
    };
    unsigned least = ~0u;  // of twice the bits of what this thread stages, less one: zeros are the largest
    char* const my_stage = stage + (my_piece / 4) * 96 + (my_piece % 4) * 8;
    auto store_pass = [&](const v4f& from, int first, int buffer) {  // without a branch: what is no pixel goes behind the last one
        v2u h, m, l;
        split_thirds(from, h, m, l);
#pragma unroll
        for (int e = 0; e < 4; ++e) least = min(least, (__float_as_uint(from[e]) << 1) - 1);
        const int at = first + my_pixel;
        char* const to = my_stage + buffer + (at < staged ? at : staged) * PITCH;
        *reinterpret_cast<v2u*>(to) = h;
        *reinterpret_cast<v2u*>(to + 32) = m;
        *reinterpret_cast<v2u*>(to + 64) = l;
    };
    load_batch(0, 0);
#pragma unroll
    for (int u = 0; u < 3; ++u) request(u, w_at + u * kTapBytes);
    float par[kParams];
    load_parameters(p, kb0 * 32 + lane, par);
    // the wave's pixels: their place in the staged rows, and in the output
    const char* b_at[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        const int at = (side * NT + n) * 32 + (lane & 31);
        const auto w = q.list.where<1>(run0 + at, p.out_h, p.out_w);
        if (part == 0) pixels[at] = w.pix;
        b_at[n] = stage + ((w.row - first_row) * q.list.staged_cols + w.x) * PITCH + half * 16;
    }
    const int tap_row = q.list.staged_cols * PITCH;
    v16f acc[MT][NT], low[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[m][n][e] = low[m][n][e] = 0.f;
    auto product = [&](int u, const v8bf (&b)[NT][3], int ta, int tb, v16f (&to)[MT][NT]) {
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int n = 0; n < NT; ++n) to[m][n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[u][m][ta], b[n][tb], to[m][n], 0, 0, 0);
    };
    for (int first = 0;;) {
#pragma unroll
        for (int i = 0; i < BATCH; ++i)
            if (first + i * PASS < staged) store_pass(x[i], first + i * PASS, 0);
        first += BATCH * PASS;
        if (first >= staged) break;
        load_batch(first, 0);
    }
#pragma unroll
    for (int i = 0; i < kParams; ++i)
        if (lane < MT * 32) params[i * MT * 32 + lane] = par[i];  // (every wave the same)
    __syncthreads();

    // A chunk's products; NEXT: and under those of each of its steps a batch of the next chunk's pixels on their way into the other buffer.
    int step = part, here = 0;
    auto products = [&](int chunk, auto next) {
        constexpr bool NEXT = decltype(next)::value;
#pragma unroll 1
        for (int s = part; s < CS && (NEXT || step < p.csteps); s += WK, step += WK) {
            const bool more = step + WK < p.csteps;  // (a next chunk need not have a step for every wave)
            const int first = s / WK * (BATCH * PASS);
            if constexpr (NEXT) load_batch(first, chunk + 1);
            v8bf b[3][NT][3];
            auto fetch = [&](v8bf (&to)[NT][3], int at) {
#pragma unroll
                for (int n = 0; n < NT; ++n)
#pragma unroll
                    for (int t = 0; t < 3; ++t) to[n][t] = *reinterpret_cast<const v8bf*>(b_at[n] + at + t * 32);
            };
            auto tap = [&](int u, const v8bf (&now)[NT][3], int w_next) {
                product(u, now, 2, 1, low);
                product(u, now, 1, 2, low);
                product(u, now, 2, 0, low);
                product(u, now, 0, 2, low);
                product(u, now, 1, 1, low);
                product(u, now, 1, 0, low);
                product(u, now, 0, 1, low);
                product(u, now, 0, 0, acc);
                request(u, w_next);
                __builtin_amdgcn_sched_barrier(0);
            };
            auto next_step = [&]() {  // what is requested from here on belongs to the next step
                w_at += WK * kStepBytes;
#pragma unroll
                for (int m = 0; m < MT; ++m) woff[m] = more ? woff[m] : kOutOfRange;
            };
            int row_at = here + s * 96;
            fetch(b[0], row_at);
            if constexpr (NEXT) {
#pragma unroll
                for (int i = 0; i < 9; ++i) {
                    if (i < 8) fetch(b[(i + 1) % 3], row_at + (i + 1) / 3 * tap_row + (i + 1) % 3 * PITCH);
                    __builtin_amdgcn_sched_barrier(0);  // (the reads would sink to the next tap's first product)
                    if (i == 6) next_step();
                    if (i >= 3) {
#pragma unroll
                        for (int k = (i - 3) * PER_TAP; k < (i - 2) * PER_TAP && k < BATCH; ++k) store_pass(x[k], first + k * PASS, q.buffer_b - here);
                    }
                    tap(i % 3, b[i % 3], w_at + (i < 6 ? i + 3 : i - 6) * kTapBytes);
                }
            } else {  // the last chunk, often the only one: a filter row at a time, since no cache has seen a launch's code yet
#pragma unroll 1
                for (int r = 0; r < 3; ++r) {
                    int w_next = w_at + (r + 1) * (3 * kTapBytes), row_next = row_at + tap_row;
                    if (r == 2) {
                        next_step();
                        w_next = w_at;
                        row_next = row_at;  // (what is read there is not used)
                    }
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        fetch(b[(c + 1) % 3], c == 2 ? row_next : row_at + (c + 1) * PITCH);
                        __builtin_amdgcn_sched_barrier(0);
                        tap(c, b[c], w_next + c * kTapBytes);
                    }
                    row_at = row_next;
                }
            }
        }
    };
#pragma unroll 1
    for (int chunk = 0; chunk + 1 < q.chunks; ++chunk) {
        products(chunk, std::true_type{});
        for (int first = CS / WK * (BATCH * PASS); first < staged; first += BATCH * PASS) {
            load_batch(first, chunk + 1);
#pragma unroll
            for (int i = 0; i < BATCH; ++i)
                if (first + i * PASS < staged) store_pass(x[i], first + i * PASS, q.buffer_b - here);
        }
        here = q.buffer_b - here;
        __syncthreads();
    }
    products(q.chunks - 1, std::false_type{});

    v4f res[Tail<MT, NT, WK>::UNITS];
    load_shortcut<MT, NT, WK>(p, pixels, kb0, part, side, lane, res);
    __syncthreads();  // the staged pixels are no longer read
    char* const red = stage + side * (WK * BLOCKS * 4096);
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[m][n] += low[m][n];
    put_sums<MT, NT>(acc, red, part, lane);
    // The loads are waited for here. In finish_tile's loop the wait would take its own stores along: one counter counts both, and a unit would
    // last 1000 cycles.
#pragma unroll
    for (int u = 0; u < Tail<MT, NT, WK>::UNITS; ++u) asm volatile("" : "+v"(res[u]));
    __syncthreads();
    bool missing = least < (kLeast << 1) - 1;  // what thirds do not hold: what this thread staged, or a sum it finishes
    auto any_missing = [&]() {
        if (missing) *again = 1;
        __syncthreads();
        return *again != 0;
    };
    bool found = false;
    if (q.in_place) {  // nothing may be stored before it is known, then: a second time reads the shortcut again
        for (int i = threadIdx.x * 16; i < WAVES * BLOCKS * 4096; i += THREADS * 16) {
            const v4f t = *reinterpret_cast<const v4f*>(stage + i);
#pragma unroll
            for (int e = 0; e < 4; ++e) missing |= no_sum(t[e]);
        }
        found = any_missing();
    }
    if (!found) {
        if (Tail<MT, NT, WK>::owner(part)) missing |= finish_tile<MT, NT, WK, SLOW>(q, pixels, params, red, kb0, part, side, lane, res);
        if (!q.in_place) found = any_missing();
    }
    if (__builtin_expect(found, 0)) {
#ifdef __HIP_DEVICE_COMPILE__
        const auto* const args = (const ThirdsParams*)__builtin_amdgcn_kernarg_segment_ptr();
#else
        const auto* const args = &q;
#endif
        again_with_floats<MT, NT, WK, SLOW>(args, pixels, params, red, kb0, part, side, lane);
    }
}

std::mutex g_attr_mutex;

// A launch's form and strips.
struct Plan {
    int form = -1;
    exhip_strips strips;
};

constexpr int kForms = 5;
struct Shape {
    int mt, nt, wk, wp, cs, occ;  // conv3x3_thirds_kernel's template arguments
};
constexpr Shape kForm[kForms] = {{1, 1, 4, 1, 4, 3}, {1, 1, 8, 1, 8, 2}, {1, 1, 2, 2, 2, 3}, {1, 1, 1, 4, 1, 3}, {2, 1, 2, 2, 2, 2}};

struct Sizes {
    int run, pitch, waves;
    explicit Sizes(const Shape& f) : run(32 * f.nt * f.wp), pitch(f.cs * 96 + 16), waves(f.wk * f.wp), f_(f) {}
    int table_bytes(int staged) const { return ((run + kParams * f_.mt * 32 + 4 + staged) * 4 + 15) / 16 * 16; }
    int lds(int staged, int buffers) const { return table_bytes(staged) + std::max((staged + 1) * pitch * buffers, waves * f_.mt * f_.nt * 4096); }
    // staged pixels with which as many of `items` groups share a CU as its registers allow. With room for three where a CU gets one, strips were so narrow that the columns
    // a map does not have made a second round: 128 -> 128 at 3 x 26 x 26 264 groups for 256, 10.1 us, now 8.2; 512 -> 512 at 3 x 13 x 13 29.5, now 24.8.
    int most(int buffers, long long items) const {
        const int resident = (int)std::min<long long>(std::max(f_.occ * 4 / waves, 1), (items + 255) / 256);
        return (kLdsLimit / resident - table_bytes(0) - 16 - pitch * buffers) / (pitch * buffers + 4);
    }

private:
    const Shape f_;
};

// The form that a model of the launch says is shortest, in microseconds: 2.5 for the launch; per round of groups on 256 CUs 1.5 for a group's
// start, 0.2 for every four channels of a pixel that a thread finishes and 0.09 for every chunk; the products at 0.019 each, all of a SIMD's or
// a group's where it is alone; or the weights at 14.6 TB/s where that is longer. Its choice is 1 % slower than the fastest of these forms on average, over 62 layers
// from 1 x 11 x 11 to 37 GFLOP.
int choose_form(const F32Params& p, long long pixels, int kblocks) {
    int best = 0;
    double best_cost = 0;
    for (int i = 0; i < kForms; ++i) {
        const Shape& f = kForm[i];
        const int waves = f.wk * f.wp, blocks = f.mt * f.nt, steps = (p.csteps + f.wk - 1) / f.wk, units = std::max(1, blocks * 4 / f.wk);
        const int resident = std::max(1, f.occ * 4 / waves);
        const long long items = (pixels + 32 * f.nt * f.wp - 1) / (32 * f.nt * f.wp) * ((kblocks + f.mt - 1) / f.mt), each = (items + 255) / 256;
        const double products = steps * 9 * blocks * 8 * 0.0191, rounds = (double)((each + resident - 1) / resident);
        const double time = rounds * (1.5 + 0.2 * units + 0.09 * ((p.csteps + f.cs - 1) / f.cs - 1)) + std::max(each * (waves / 4) * products, rounds * products);
        const double cost = std::max(time, (double)items * f.mt * p.csteps * kStepBytes / 14.6e6);
        if (i == 0 || cost < best_cost) {
            best_cost = cost;
            best = i;
        }
    }
    return best;
}

// A thread keeps the plans of its last layers: the search is 1 to 2 us, half of what a launch costs the host.
const Plan& plan_of(const F32Params& p, long long images, int kblocks, int tile) {
    struct Entry {
        long long images = -1;
        int h, w, csteps, kblocks, tile;
        Plan plan;
    };
    static thread_local Entry cache[64];
    Entry& e = cache[(unsigned)(p.out_h * 31 + p.out_w * 7 + p.csteps * 5 + kblocks * 3 + (int)images) % 64];
    if (e.images != images || e.h != p.out_h || e.w != p.out_w || e.csteps != p.csteps || e.kblocks != kblocks || e.tile != tile) {
        e = Entry();
        e.h = p.out_h; e.w = p.out_w; e.csteps = p.csteps; e.kblocks = kblocks; e.tile = tile;
        const int chosen = tile > 0 ? std::min(tile, kForms) - 1 : choose_form(p, (long long)p.out_h * p.out_w * images, kblocks);
        // Maps of a few pixels stage up to nine for each. LDS holds nine times the first form's 32 pixels once, but not twice: of maps of one pixel every second
        // lane has one then (16 images stage 192 pixels).
        for (int tries = 0; tries < 3; ++tries) {
            const int form = tries ? 0 : chosen, buffers = p.csteps > kForm[form].cs ? 2 : 1;
            const Sizes s(kForm[form]);
            const long long groups = (kblocks + kForm[form].mt - 1) / kForm[form].mt, items = ((long long)p.out_h * p.out_w * images + s.run - 1) / s.run * groups;
            e.plan.form = form;
            e.plan.strips = exhip_choose_strips(p.out_h, p.out_w, 1, images, s.run, s.most(buffers, items), groups, tries == 2);
            if (s.lds(e.plan.strips.staged, buffers) <= kLdsLimit) break;
        }
        e.images = images;
    }
    return e.plan;
}

template <int FORM, bool SLOW>
int go(exhip_ctx* ctx, ThirdsParams& q, const Plan& plan, long long images, int kblocks) {
    constexpr Shape f = kForm[FORM];
    const Sizes s(f);
    F32Params& p = q.f;
    q.chunks = (p.csteps + f.cs - 1) / f.cs;
    const int lds = s.lds(plan.strips.staged, q.chunks > 1 ? 2 : 1);
    EXHIP_REQUIRE(lds <= kLdsLimit, "conv: %d pixels to stage", plan.strips.staged);
    q.list.set(plan.strips, p.out_h, 1, images);
    q.table_b = s.table_bytes(plan.strips.staged);
    q.buffer_b = (plan.strips.staged + 1) * s.pitch;
    const long long groups = (kblocks + f.mt - 1) / f.mt, items = plan.strips.tiles * groups;
    EXHIP_REQUIRE(items < (1ll << 31) - 4, "conv: grid too large");
    p.items = (unsigned)items;
    p.tiles_fast = p.w_bytes > (4u << 20) && p.w_bytes > p.x_bytes;  // (conv_f32_kernel)
    p.fast = (unsigned)(p.tiles_fast ? plan.strips.tiles : groups);
    q.by_fast.set(p.fast);
    auto kernel = conv3x3_thirds_kernel<f.mt, f.nt, f.wk, f.wp, f.cs, f.occ, SLOW>;
    {
        static unsigned long long attr_set = 0;
        std::lock_guard<std::mutex> lock(g_attr_mutex);
        const unsigned long long bit = 1ull << (ctx->device & 63);
        if (!(attr_set & bit)) {
            EXHIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kLdsLimit));
            attr_set |= bit;
        }
    }
    hipLaunchKernelGGL(kernel, dim3(p.items), dim3(64 * f.wk * f.wp), lds, ctx->stream, q);
    EXHIP_LAUNCH_CHECK();
    return 0;
}

// A weight's thirds. An infinity is its own first third; what would round up to an infinity is cut off; what thirds do not hold is kept whole.
__host__ __device__ inline void split_weight(float x, uint16_t (&out)[3]) {
    const unsigned whole = __builtin_bit_cast(unsigned, x), size = whole & 0x7fffffffu;
    if ((size > 0 && size < kLeast) || size > 0x7f800000u) {
        out[0] = kWhole;
        out[1] = (uint16_t)(whole >> 16);
        out[2] = (uint16_t)whole;
        return;
    }
    for (int t = 0; t < 3; ++t) {
        const unsigned b = __builtin_bit_cast(unsigned, x), r = b + 0x7fffu + (b >> 16 & 1);
        const bool finite = (b & 0x7f800000u) != 0x7f800000u;
        const unsigned third = finite && (r & 0x7f800000u) != 0x7f800000u ? r >> 16 : b >> 16;
        out[t] = (uint16_t)third;
        x = finite ? x - __builtin_bit_cast(float, third << 16) : 0.f;
    }
}

typedef unsigned v8w __attribute__((ext_vector_type(8)));
typedef float v8f __attribute__((ext_vector_type(8)));
typedef uint16_t v8s __attribute__((ext_vector_type(8)));

// Eight channels' nine taps to where a lane has them, [tap][third] 1 KiB each: eight channels at a time where all weights are zeros or between 2^-103 and what rounds
// up to an infinity.
__attribute__((always_inline)) inline bool split_finite(const float* src, char* to) {
    v8w w[9], t[8];  // [tap]: the rows of eight taps turned over, and the ninth
    for (int i = 0; i < 8; ++i) {
        memcpy(&w[i], src + i * 9, 32);
        memcpy(reinterpret_cast<char*>(&w[8]) + i * 4, src + i * 9 + 8, 4);
    }
    for (int i = 0; i < 8; i += 2) {
        t[i] = __builtin_shufflevector(w[i], w[i + 1], 0, 8, 2, 10, 4, 12, 6, 14);
        t[i + 1] = __builtin_shufflevector(w[i], w[i + 1], 1, 9, 3, 11, 5, 13, 7, 15);
    }
    for (int i = 0; i < 8; i += i % 4 == 1 ? 3 : 1) {
        w[i] = __builtin_shufflevector(t[i], t[i + 2], 0, 1, 8, 9, 4, 5, 12, 13);
        w[i + 2] = __builtin_shufflevector(t[i], t[i + 2], 2, 3, 10, 11, 6, 7, 14, 15);
    }
    for (int i = 0; i < 4; ++i) {
        t[i] = __builtin_shufflevector(w[i], w[i + 4], 0, 1, 2, 3, 8, 9, 10, 11);
        t[i + 4] = __builtin_shufflevector(w[i], w[i + 4], 4, 5, 6, 7, 12, 13, 14, 15);
    }
    v8w high = 0, least = ~0u;
    for (int tap = 0; tap < 9; ++tap) {
        if (tap < 8) w[tap] = t[tap];
        high |= (w[tap] & 0x7fffffffu) + 0x808000u;  // the sign bit from 0x7f7f8000 on
        least = __builtin_elementwise_min(least, (w[tap] << 1) - 1);
    }
    for (int i = 0; i < 8; ++i)
        if (high[i] & 0x80000000u || least[i] < (kLeast << 1) - 1) return false;
    for (int tap = 0; tap < 9; ++tap) {
        v8f x = __builtin_bit_cast(v8f, w[tap]);
        for (int third = 0; third < 3; ++third) {
            v8w b = __builtin_bit_cast(v8w, x);
            b = (b + 0x7fffu + (b >> 16 & 1)) & 0xffff0000u;  // to the nearest, ties to even
            x -= __builtin_bit_cast(v8f, b);
            const v8s out = __builtin_convertvector(b >> 16, v8s);
            memcpy(to + (tap * 3 + third) * 1024, &out, 16);
        }
    }
    return true;
}

// The output channel that lane rr of either half has in a block.
__host__ __device__ inline int lane_channel(int kb, int lane) {
    const int rr = lane % 32;
    return kb * 32 + (rr / 4 % 2) * 16 + rr / 8 * 4 + rr % 4;
}

// One step's weights of a 32-channel block.
__attribute__((always_inline)) inline void pack_step(const float* w, int C, int K, int kb, int j, char* to) {
    for (int lane = 0; lane < 64; ++lane) {
        const int k = lane_channel(kb, lane);
        const float* const src = w + ((size_t)k * C + j * 16 + lane / 32 * 8) * 9;
        if (k < K && split_finite(src, to + lane * 16)) continue;
        for (int i = 0; i < 72; ++i) {
            uint16_t thirds[3] = {};
            if (k < K) split_weight(src[i], thirds);
            for (int t = 0; t < 3; ++t) memcpy(to + (i % 9 * 3 + t) * 1024 + lane * 16 + i / 9 * 2, &thirds[t], 2);
        }
    }
}
#ifndef __HIP_DEVICE_COMPILE__
__attribute__((target("avx2"))) void pack_step_avx2(const float* w, int C, int K, int kb, int j, char* to) { pack_step(w, C, K, kb, j, to); }
#endif
void pack_step_any(const float* w, int C, int K, int kb, int j, char* to) { pack_step(w, C, K, kb, j, to); }

}  // namespace

bool exhip_conv_f32_thirds(const exhip_conv_desc* d) {
    return d->kh == 3 && d->kw == 3 && d->sh == 1 && d->c % 16 == 0 && (long long)((d->k + 31) / 32) * (d->c / 16) * kStepBytes < (1ll << 31);
}

size_t exhip_conv_f32_thirds_bytes(const exhip_conv_desc* d) { return (size_t)((d->k + 31) / 32) * (d->c / 16) * kStepBytes; }

// [32-channel block][16 channels][tap][third][lane][8 bfloat16]: lane rr of either half has the output channel that conv_f32.hip's packing gives
// it, and eight neighbouring input channels. .8 ns a weight (whole floats 1.0).
void exhip_conv_f32_thirds_pack(const exhip_conv_desc* d, const float* w, void* out) {
    const int C = d->c, K = d->k, steps = C / 16, blocks = (K + 31) / 32;
    auto step = pack_step_any;
#ifndef __HIP_DEVICE_COMPILE__
    if (__builtin_cpu_supports("avx2")) step = pack_step_avx2;
#endif
    for (int kb = 0; kb < blocks; ++kb)
        for (int j = 0; j < steps; ++j) step(w, C, K, kb, j, static_cast<char*>(out) + (size_t)(kb * steps + j) * kStepBytes);
}

// The same on the device: a wave a step and block, a lane its eight channels' taps. A network's first call uploads two thirds of the bytes then, and the host, which takes .5
// to 2 ms for a layer of 512 -> 512 whose weights no cache holds, has nothing to pack (first call of the text detector 9.2 -> 5.1 ms, of the float32 detector 9.7 -> 8.8).
__global__ __launch_bounds__(64) void pack_thirds_kernel(const float* __restrict__ w, char* __restrict__ out, int C, int K, int steps) {
    const int lane = threadIdx.x, kb = (int)blockIdx.x / steps, j = (int)blockIdx.x - kb * steps, k = lane_channel(kb, lane);
    const float* const src = w + ((size_t)k * C + j * 16 + lane / 32 * 8) * 9;
    char* const to = out + (size_t)blockIdx.x * kStepBytes + lane * 16;
#pragma unroll
    for (int tap = 0; tap < 9; ++tap) {
        v4u words[3] = {};
        if (k < K) {
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                uint16_t thirds[3];
                split_weight(src[c * 9 + tap], thirds);
#pragma unroll
                for (int t = 0; t < 3; ++t) words[t][c / 2] |= (unsigned)thirds[t] << (c % 2 * 16);
            }
        }
#pragma unroll
        for (int t = 0; t < 3; ++t) *reinterpret_cast<v4u*>(to + (tap * 3 + t) * 1024) = words[t];
    }
}

int exhip_conv_f32_thirds_pack_device(exhip_ctx* ctx, const exhip_conv_desc* d, const float* w, void* out) {
    const int steps = d->c / 16, blocks = (d->k + 31) / 32;
    hipLaunchKernelGGL(pack_thirds_kernel, dim3((unsigned)(blocks * steps)), dim3(64), 0, ctx->stream, w, static_cast<char*>(out), d->c, d->k, steps);
    EXHIP_LAUNCH_CHECK();
    return 0;
}

int exhip_conv_f32_thirds_run(exhip_ctx* ctx, const F32Launch& launch) {
    ThirdsParams q = {};
    q.f = *static_cast<const F32Params*>(launch.params);
    F32Params& p = q.f;
    q.plain = p.y && !p.y_nchw && p.layout == EXHIP_PLACE_ROWS && p.vector_rows && p.act <= 1 && !p.bn_a && !p.post_op && !(p.residual && p.residual_last);
    q.floor = p.act == 1 ? 0.f : -INFINITY;
    q.post_floor = p.post_relu ? 0.f : -INFINITY;
    const bool slow = p.act == 4 || p.act == 5;
    const size_t res_pixels = (size_t)(p.pixels >> 2 * p.res_shift), y_pixels = (size_t)p.pixels * (p.layout == EXHIP_PLACE_SHUFFLED ? 4 : 1);
    q.in_place = p.residual && p.y && p.residual < p.y + y_pixels * (unsigned)p.kstride && p.y < p.residual + res_pixels * (unsigned)p.rstride;
    const Plan plan = plan_of(p, launch.images, launch.blocks, slow ? 1 : g_exhip_options.f32_tile);
    switch (plan.form) {
    case 0: return slow ? go<0, true>(ctx, q, plan, launch.images, launch.blocks) : go<0, false>(ctx, q, plan, launch.images, launch.blocks);
    case 1: return go<1, false>(ctx, q, plan, launch.images, launch.blocks);
    case 2: return go<2, false>(ctx, q, plan, launch.images, launch.blocks);
    case 3: return go<3, false>(ctx, q, plan, launch.images, launch.blocks);
    default: return go<4, false>(ctx, q, plan, launch.images, launch.blocks);
    }
}
