// conv_f32_kernel: the float32 convolution, any filter, stride and padding, on NHWC input with v_mfma_f32_32x32x2_f32. (3x3 layers at stride 1
// of whole 16-channel steps run in conv_f32_thirds.hip.)
//
// float32 products run at a sixteenth of the half-precision rate (157 TFLOP/s), so operands are cheap next to the
// arithmetic: one 32-byte step of a 64-channel x 32-pixel wave tile fetches 3 KiB for 512 matrix cycles. Nothing is staged
// therefore: a wave owns 32 * NT output pixels x 32 * MT output channels and loads its fragments straight into registers,
// 16 bytes per lane and step -- the weights from a packing in which a 32-channel block is one contiguous stream, the
// pixels from the NHWC rows around each output pixel, taps outside the image reading zeros. The pixels of all images form
// one list, so ragged maps waste no lanes. No barrier in the main loop, no tile geometry, no patch to plan.
//
// What bounds it otherwise is a small launch: a 3x3 layer of 64 channels on one 56 x 56 map is 98 wave tiles for 1024 SIMDs,
// each with a chain of 72 steps. WK waves of a group therefore share a tile: each reduces its run of the steps, the parts are
// added through LDS in a fixed order (the same bits every time) and the waves share the tile's blocks in the epilogue.
//
// Arithmetic: float32 products and sums, bias, activation, the optional shortcut in front of or behind the layers behind the
// convolution, BatchNorm, activation layer.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <type_traits>

#include "conv_f32.h"
#include "conv_f32_epilogue.h"
#include "pack.h"
#include "pair.h"

namespace {

// A view of a pixel-major float tensor from pixel `first` and channel ch0 on, `rows` pixels long.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_view(const float* base, unsigned first, int stride, int ch0, int rows) {
    float* p = const_cast<float*>(base) + (size_t)first * (unsigned)stride + ch0;
    return __builtin_amdgcn_make_buffer_rsrc(p, 0, (rows * stride - ch0) * 4, kRsrcWord3);
}

template <int MT>
__device__ __forceinline__ void read16(const char* lds, int which, int m, int half, float (&v)[16]) {
    const v4f* src = reinterpret_cast<const v4f*>(lds + (which * MT * 32 + m * 32 + half * 16) * 4);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const v4f t = src[q];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[q * 4 + e] = t[e];
    }
}

template <int OP>
__device__ __forceinline__ void unary16(float (&v)[16], float alpha, float beta) {
#pragma unroll
    for (int e = 0; e < 16; ++e) v[e] = unary_value<OP>(v[e], alpha, beta);
}
__device__ __forceinline__ void relu16(float (&v)[16]) {
#pragma unroll
    for (int e = 0; e < 16; ++e) v[e] = (0.f > v[e]) ? 0.f : v[e];
}

constexpr int kTilePitch = 128 + 16;      // one pixel's 32 channels and padding
constexpr int wave_lds(int mt) { return kParams * mt * 32 * 4 + 32 * kTilePitch; }

// One 32-pixel x 32-channel block: lane = pixel (lane & 31) and sixteen neighbouring channels. Straight code per layer kind
// under wave-uniform branches; what is not taken is not fetched.
template <int MT, bool SLOW>
__device__ __forceinline__ void epilogue_block(const F32Params& p, const v16f& acc, unsigned first, int kb, int m, int lane, char* lds) {
    const int half = lane >> 5, row = lane & 31, ch0 = kb * 32 + half * 16;
    if (first >= p.pixels || kb * 32 >= p.k_end) return;
    const int rows = p.pixels - first < 32 ? (int)(p.pixels - first) : 32;
    char* const tile = lds + kParams * MT * 32 * 4;
    float v[16], t[16], res[16];
    // where the lane's pixel lies: its image and the pixel inside it, for the forms that place pixels or read them elsewhere
    const unsigned per_image = (unsigned)(p.out_h * p.out_w), pix = first + row;
    unsigned img = 0, in_image = 0;
    if (p.res_shift || p.y_nchw || p.layout != EXHIP_PLACE_ROWS) {
        img = exhip_divide(pix, per_image, p.image_magic, p.image_shift);
        in_image = pix - img * per_image;
    }
    if (p.residual) {
        unsigned from = pix;
        if (p.res_shift) {
            const unsigned oy = exhip_divide(in_image, (unsigned)p.out_w, p.width_magic, p.width_shift), ox = in_image - oy * (unsigned)p.out_w;
            from = (img * ((unsigned)p.out_h >> p.res_shift) + (oy >> p.res_shift)) * ((unsigned)p.out_w >> p.res_shift) + (ox >> p.res_shift);
        }
        const float* const src = p.residual + (size_t)from * (unsigned)p.rstride + ch0;
        if (p.vector_rows) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                v4f r = {0.f, 0.f, 0.f, 0.f};
                if (row < rows && ch0 + q * 4 < p.K) r = reinterpret_cast<const v4f*>(src)[q];
#pragma unroll
                for (int e = 0; e < 4; ++e) res[q * 4 + e] = r[e];
            }
        } else {
#pragma unroll
            for (int e = 0; e < 16; ++e) res[e] = row < rows && ch0 + e < p.K ? src[e] : 0.f;
        }
    }
    read16<MT>(lds, 0, m, half, t);
#pragma unroll
    for (int e = 0; e < 16; ++e) v[e] = acc[e] + t[e];
    if (p.act == 1) relu16(v);
    if constexpr (SLOW) {  // double-precision functions: through LDS, one value at a time, so that their registers are needed once
        float* const own = reinterpret_cast<float*>(tile) + (row * kTilePitch / 4 + half * 16);
#pragma unroll
        for (int e = 0; e < 16; ++e) own[e] = v[e];
#pragma unroll 1
        for (int e = 0; e < 16; ++e) own[e] = exhip_act(own[e], p.act);
#pragma unroll
        for (int e = 0; e < 16; ++e) v[e] = own[e];
    } else if (p.act == 3) {
#pragma unroll
        for (int e = 0; e < 16; ++e) v[e] = exhip_act(v[e], 3);
    }
    if (p.residual && !p.residual_last) {
#pragma unroll
        for (int e = 0; e < 16; ++e) v[e] += res[e];
    }
    if (p.post_relu) relu16(v);
    if (p.bn_a) {
        read16<MT>(lds, 2, m, half, t);
        float b[16];
        read16<MT>(lds, 3, m, half, b);
#pragma unroll
        for (int e = 0; e < 16; ++e) v[e] = __builtin_fmaf(b[e], v[e], t[e]);
        if (p.bn_relu) relu16(v);
    }
    switch (p.post_op) {
    case 0: break;
    case 1 + EXHIP_UNARY_HARDSWISH: unary16<0>(v, p.alpha, p.beta); break;
    case 1 + EXHIP_UNARY_LEAKYRELU: unary16<1>(v, p.alpha, p.beta); break;
    case 1 + EXHIP_UNARY_HARDSIGMOID: unary16<3>(v, p.alpha, p.beta); break;
    case 1 + EXHIP_UNARY_CLIP: unary16<4>(v, p.alpha, p.beta); break;
    default:
        read16<MT>(lds, 1, m, half, t);
#pragma unroll
        for (int e = 0; e < 16; ++e) v[e] = v[e] >= 0.f ? v[e] : t[e] * v[e];
    }
    if (p.residual && p.residual_last) {
#pragma unroll
        for (int e = 0; e < 16; ++e) v[e] += res[e];
    }
    if (p.y) {
        if (kb * 32 + 32 > p.K) {  // pad channels hold zeros
#pragma unroll
            for (int e = 0; e < 16; ++e)
                if (ch0 + e >= p.K) v[e] = 0.f;
        }
        if (p.vector_rows || p.layout == EXHIP_PLACE_GROUPED) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const v4f o = {v[q * 4], v[q * 4 + 1], v[q * 4 + 2], v[q * 4 + 3]};
                *reinterpret_cast<v4f*>(tile + row * kTilePitch + half * 64 + q * 16) = o;
            }
        }
        if (p.layout == EXHIP_PLACE_GROUPED) {
            // y[img][group][pixel][member]: a half-wave writes the block's 32 channels of one pixel, runs of neighbouring floats
            const int ch = kb * 32 + row, g = ch / p.group, member = ch - g * p.group;
            const unsigned lane_at = img * (unsigned)p.K * per_image + in_image * (unsigned)p.group;
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                const int srow = j * 2 + half;
                const unsigned at = (unsigned)__builtin_amdgcn_ds_bpermute(srow * 4, (int)lane_at) + (unsigned)g * per_image * (unsigned)p.group + member;
                if (srow < rows && ch < p.K) p.y[at] = *reinterpret_cast<const float*>(tile + srow * kTilePitch + row * 4);
            }
        } else if (p.layout == EXHIP_PLACE_SHUFFLED) {
            // channel pos * group + k of pixel (y, x) is channel k of pixel (2 y + pos / 2, 2 x + pos % 2) of a map twice as large
            const unsigned oy = exhip_divide(in_image, (unsigned)p.out_w, p.width_magic, p.width_shift), ox = in_image - oy * (unsigned)p.out_w;
            const unsigned corner = (img * 2 * (unsigned)p.out_h + 2 * oy) * 2 * (unsigned)p.out_w + 2 * ox;
            if (p.vector_rows) {  // whole blocks belong to one of the four
                const int pos = kb * 32 / p.group, k0 = kb * 32 - pos * p.group;
                const unsigned step = (unsigned)(pos >> 1) * 2 * (unsigned)p.out_w + (pos & 1);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int srow = j * 8 + (lane >> 3);
                    const unsigned to = (unsigned)__builtin_amdgcn_ds_bpermute(srow * 4, (int)corner) + step;
                    if (srow < rows)
                        *reinterpret_cast<v4f*>(p.y + (size_t)to * (unsigned)p.kstride + k0 + (lane & 7) * 4) =
                            *reinterpret_cast<const v4f*>(tile + srow * kTilePitch + (lane & 7) * 16);
                }
            } else if (row < rows) {
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const int pos = (ch0 + e) / p.group, k = ch0 + e - pos * p.group;
                    if (ch0 + e < p.K)
                        p.y[(size_t)(corner + (unsigned)(pos >> 1) * 2 * (unsigned)p.out_w + (pos & 1)) * (unsigned)p.kstride + k] = v[e];
                }
            }
        } else {
            const __amdgpu_buffer_rsrc_t yr = rows_view(p.y, first, p.kstride, kb * 32, rows);
            if (p.vector_rows) {  // through LDS: eight neighbouring lanes write one pixel's 128 bytes
                const int scol = (lane & 7) * 16;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int srow = j * 8 + (lane >> 3);
                    const v4u o = *reinterpret_cast<const v4u*>(tile + srow * kTilePitch + scol);
                    const bool in = srow < rows && scol < (p.k_end - kb * 32) * 4;
                    __builtin_amdgcn_raw_buffer_store_b128(o, yr, in ? srow * p.kstride * 4 + scol : (int)kOutOfRange, 0, 0);
                }
            } else {
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v[e]), yr,
                                                          row < rows && ch0 + e < p.k_end ? (row * p.kstride + half * 16 + e) * 4 : (int)kOutOfRange, 0, 0);
            }
        }
    }
    if (p.y_nchw && row < rows) {  // 32 neighbouring pixels of a channel per store instruction and half-wave
        float* const dst = p.y_nchw + ((size_t)img * p.K + ch0) * per_image + in_image;
#pragma unroll
        for (int e = 0; e < 16; ++e)
            if (ch0 + e < p.K) dst[(size_t)e * per_image] = v[e];
    }
}

// R: requested steps in flight. PAIRS: the pixels in 64-byte pieces, two steps at a time.
template <int MT, int NT, int WK>
struct F32Shape {
    static constexpr int WAVES = WK > 4 ? WK : 4, ITEMS = WAVES / WK;  // tiles per group
    static constexpr int BLOCKS = MT * NT;
    // A wave of a split tile finishes a block, and stores its rows through LDS, or where that leaves every block to four waves or more a
    // quarter of one (four channels a lane), and stores from registers. Halves from registers fill lines in pieces of 32 bytes, and launches
    // of two waves a block are still large: 64 -> 64 3x3 at 24 x 40 x 40 33.8 us in halves, 28.9 in blocks, 128 -> 128 at 4 x 80 x 80 73.7 and
    // 64.3, 1x1 64 -> 64 at 8 x 80 x 80 12.9 and 11.1.
    static constexpr bool ROWS = WK == 1 || WK < 4 * BLOCKS;
    static constexpr int OWNERS = WK > 1 ? BLOCKS : 1;              // ROWS: waves of a tile that finish a block
    static constexpr int RED = WK > 1 ? WAVES * BLOCKS * 4096 : 0;  // the waves' partial sums
    static constexpr int LDS = RED + (ROWS ? ITEMS * OWNERS * wave_lds(MT) : 0);
    static_assert(WK == 1 || OWNERS <= WK, "a wave finishes at most one block");
};
// (the kernel's group `bid` of `groups`)
template <int MT, int NT, int WK, int R, int MODE, bool PAIRS, bool SLOW>
__device__ __forceinline__ void f32_group(const F32Params& p, char* lds_all, unsigned bid, unsigned groups) {
    typedef F32Shape<MT, NT, WK> Shape;
    constexpr int ITEMS = Shape::ITEMS, BLOCKS = Shape::BLOCKS, OWNERS = Shape::OWNERS, RED = Shape::RED;
    constexpr bool ROWS = Shape::ROWS;
    constexpr int QUADS = ROWS ? 4 : 1, V = 4 * QUADS;            // WK > 1: quarters of a block that a wave finishes
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int part = wave % WK;
    // workgroup ids are dealt round-robin to the 8 XCDs: give each XCD one contiguous run of items. Either the channel groups of
    // a pixel tile run fastest, and an XCD reads its share of the pixels and all weights, or the pixel tiles do (tiles_fast)
    // and it reads its share of the weights and all pixels.
    {
        const unsigned per = groups >> 3;
        if (bid < (per << 3)) bid = (bid & 7) * per + (bid >> 3);
    }
    const unsigned item = __builtin_amdgcn_readfirstlane(bid * ITEMS + wave / WK);
    if (WK == 1 && item >= p.items) return;  // wave-uniform; that form has no barrier
    const bool on = item < p.items;
    const unsigned slow = exhip_divide(item, p.fast, p.fast_magic, p.fast_shift), fast = item - slow * p.fast;
    const unsigned tile = __builtin_amdgcn_readfirstlane(p.tiles_fast ? fast : slow);
    const int kb0 = __builtin_amdgcn_readfirstlane((int)(p.tiles_fast ? slow : fast) * MT);  // first 32-channel block

    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(p.x), 0, (int)p.x_bytes, kRsrcWord3);
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(p.wp), 0, (int)p.w_bytes, kRsrcWord3);

    // What a lane requests of the pixels. PAIRS: two steps at a time, 64 bytes of every pixel; four lanes read a pixel's, sixteen pixels a
    // load. Else a step at a time: the lane's pixel is lane & 31, its 16-byte half lane >> 5.
    constexpr int XL = PAIRS ? 2 : 1;
    static_assert(!PAIRS || R % 4 == 0, "two operand buffers take turns");
    const unsigned per_image = (unsigned)(p.out_h * p.out_w);
    const int lane_byte = (PAIRS ? lane & 3 : lane >> 5) * 16;
    unsigned xoff[NT][XL];
    int iy[NT][XL], ix[NT][XL];
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int l = 0; l < XL; ++l) {
            const unsigned pix = (tile * NT + n) * 32 + (PAIRS ? l * 16 + (lane >> 2) : lane & 31);
            const bool in = on && pix < p.pixels;
            if (MODE == kPoint && p.stride == 1) {
                xoff[n][l] = in ? pix * (unsigned)p.xs_b + lane_byte : kOutOfRange;
            } else {
                // the filter's top-left input pixel; its offset may lie in front of the tensor (padding), the taps inside the
                // image never do, and 32-bit wrap-around of the sum gives their offsets
                const unsigned img = exhip_divide(pix, per_image, p.image_magic, p.image_shift), rem = pix - img * per_image;
                const int oy = (int)exhip_divide(rem, (unsigned)p.out_w, p.width_magic, p.width_shift), ox = (int)(rem - (unsigned)oy * (unsigned)p.out_w);
                iy[n][l] = oy * p.stride - p.pad_t;
                ix[n][l] = ox * p.stride - p.pad_l;
                xoff[n][l] = (unsigned)((((int)img * p.in_h + iy[n][l]) * p.in_w + ix[n][l]) * p.xs_b + lane_byte);
                if (MODE == kPair) ix[n][l] += lane >> 5;
                if (!in) {
                    iy[n][l] = -0x40000000;
                    if (MODE == kPoint) xoff[n][l] = kOutOfRange;
                }
            }
        }
    const int s_first = p.start_s[part], steps = on ? p.start_s[part + 1] - s_first : 0;
    // the next step to request: its weights, its filter row and tap, and how far it lies behind the tap's first channel
    int w_at = s_first * 1024, r_at = p.start_r[part], q_at = p.start_q[part], c_at = p.start_c[part] * 32;
    const int w_last = (p.n_ksteps - XL) * 1024, c_end = p.csteps * 32;
    // a block past the packed ones (pad channels of a wide stride, the second half of a last pair) reads zeros
    const int wbase = kb0 * p.n_ksteps * 1024;
    unsigned woff[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) woff[m] = (kb0 + m) * 32 < p.K ? (unsigned)(m * p.n_ksteps * 1024 + lane * 16) : kOutOfRange;
    unsigned xcur[NT][XL];  // the lane's offsets at the tap, out of range where the tap lies outside the image
    auto enter_tap = [&]() {
        const int off = r_at * p.row_b + q_at * p.xs_b;
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int l = 0; l < XL; ++l) {
                const bool in = (unsigned)(iy[n][l] + r_at) < (unsigned)p.in_h && (unsigned)(ix[n][l] + q_at) < (unsigned)p.in_w &&
                                (MODE != kPair || q_at + (lane >> 5) < p.kw);
                xcur[n][l] = in ? xoff[n][l] + (unsigned)off : kOutOfRange;
            }
    };
    if constexpr (MODE == kPoint) {
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int l = 0; l < XL; ++l) xcur[n][l] = xoff[n][l];
    } else {
        enter_tap();
    }

    v16f acc[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[m][n][e] = 0.f;

    v4f a[R][MT], b[R][NT];  // a ring of requested steps
    // Requests are unconditional, so that the waits in front of the products count exactly what is in flight (behind a branch
    // the compiler has to wait for everything: 510 cycles a step instead of 420). Those past this wave's run read what lies
    // there -- the next part's operands, the last step's again -- and are not used. A step costs a handful of scalar
    // instructions; where a tap ends, a branch without memory accesses finds the next one's offsets (evaluated in every
    // step, the tap's tests stretched a step by 150 cycles where a SIMD has one wave).
    auto request = [&](int u) {  // PAIRS: steps u and u + 1, u even
#pragma unroll
        for (int l = 0; l < XL; ++l) {
#pragma unroll
            for (int m = 0; m < MT; ++m) a[u + l][m] = load4(wr, woff[m], wbase + w_at + l * 1024);
#pragma unroll
            for (int n = 0; n < NT; ++n) b[u + l][n] = load4(xr, xcur[n][l], c_at);
        }
        w_at = w_at + XL * 1024 < w_last ? w_at + XL * 1024 : w_last;
        c_at += XL * 32;
        if constexpr (MODE == kPoint) {
            c_at = c_at < c_end - XL * 32 ? c_at : c_end - XL * 32;
        } else if (c_at == c_end) {
            c_at = 0;
            q_at += MODE == kPair ? 2 : 1;
            if (q_at >= p.kw) {
                q_at = 0;
                ++r_at;
            }
            enter_tap();
        }
    };
    // PAIRS: through the wave's own LDS from four lanes a pixel to one. A CU takes 16 cycles for a load whose neighbouring lanes read
    // 64 bytes of a pixel, up to 64 for one whose lanes read pixels a power of two apart. A pixel's 16-byte columns are dealt
    // out by its number, so that neither side meets bank conflicts.
    char* const stage = lds_all + (WK > 1 ? wave * BLOCKS * 4096 : wave * wave_lds(MT) + kParams * MT * 32 * 4);
    char* const stage_in = stage + (lane >> 2) * 64 + ((lane & 3) ^ (lane >> 3 & 3)) * 16;
    const char* const stage_out = stage + (lane & 31) * 64;
    v4f x[2][2][NT];
    auto arrange = [&](int u, int to) {
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int l = 0; l < 2; ++l) *reinterpret_cast<v4f*>(stage_in + n * 2048 + l * 1024) = b[u + l][n];
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int l = 0; l < 2; ++l) x[to][l][n] = *reinterpret_cast<const v4f*>(stage_out + n * 2048 + (((2 * l + (lane >> 5)) ^ (lane >> 1 & 3)) * 16));
    };
    auto product = [&](int u, const v4f (&xb)[NT]) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int n = 0; n < NT; ++n) acc[m][n] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[u][m][e], xb[n][e], acc[m][n], 0, 0, 0);
    };
    auto step = [&](int u) {  // PAIRS: the pair, whose pixels have been arranged
        if constexpr (PAIRS) {
            product(u, x[u / 2 & 1][0]);
            product(u + 1, x[u / 2 & 1][1]);
        } else {
            product(u, b[u]);
        }
    };
#pragma unroll
    for (int u = 0; u < R / 2; u += XL) request(u);
    // WK > 1: what a wave finishes of the tile -- channels ch0 .. ch0 + V - 1 of a pixel per lane -- and their parameters;
    // ROWS: the parameters lane by lane, of the wave's MT * 32 channels
    const int quad = part * QUADS, half = lane >> 5;
    const bool owner = on && quad < 4 * BLOCKS;
    const int own_ch = (kb0 + quad / 4 % MT) * 32 + half * 16 + quad % 4 * 4;
    const unsigned own_pix = (tile * NT + quad / 4 / MT) * 32 + (lane & 31);
    constexpr int PV = ROWS ? 1 : V;
    float par[kParams][PV] = {};
    auto load_parameters = [&]() {
        const unsigned at = (unsigned)(ROWS ? kb0 * 32 + lane : own_ch) * 4;
        auto load = [&](int i, const float* src, unsigned offset, int count, int step) {
            if (!ROWS && !src) return;
            const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(src), 0, src ? count * 4 : 0, kRsrcWord3);
#pragma unroll
            for (int e = 0; e < PV; ++e) par[i][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)offset + e * step, 0, 0));
        };
        load(0, p.bias, at, p.K, 4);
        load(1, p.slope, p.slope_shared ? 0 : at, p.slope_shared ? 1 : p.K, p.slope_shared ? 0 : 4);
        load(2, p.bn_a, at, p.K, 4);
        load(3, p.bn_b, at, p.K, 4);
    };
    if (ROWS) load_parameters();
#pragma unroll
    for (int u = R / 2; u < R; u += XL) request(u);
    if constexpr (PAIRS) arrange(0, 0);
    int s = 0;
    for (; s + R < steps; s += R) {
#pragma unroll
        for (int u = 0; u < R; u += XL) {
            if constexpr (PAIRS) arrange((u + 2) % R, (u / 2 + 1) & 1);
            step(u);
            request(u);
            __builtin_amdgcn_sched_barrier(0);  // each slot is requested again as soon as its products have been issued
        }
    }
    // (the loop leaves with the last steps, at most R, requested)
    if (!ROWS && owner) load_parameters();
    char* const lds = lds_all + RED + (ROWS && part < OWNERS ? (wave / WK * OWNERS + part) * wave_lds(MT) : 0);
    if (ROWS && part < OWNERS && (MT == 2 || lane < 32)) {
#pragma unroll
        for (int i = 0; i < kParams; ++i) *reinterpret_cast<float*>(lds + (i * MT * 32 + lane) * 4) = par[i][0];
    }
#pragma unroll
    for (int u = 0; u < R; u += XL)
        if (s + u < steps) {
            if constexpr (PAIRS)
                if (u + 2 < R) arrange(u + 2, (u / 2 + 1) & 1);
            step(u);
        }
    if constexpr (WK == 1) {
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                epilogue_block<MT, SLOW>(p, acc[m][n], (tile * NT + n) * 32, kb0 + m, m, lane, lds);
                __builtin_amdgcn_sched_barrier(0);
            }
    } else {
        unsigned img = 0, in_image = 0;
        float res[V] = {}, v[V];
        if (!ROWS && owner) {
            if (p.res_shift || p.y_nchw || p.layout != EXHIP_PLACE_ROWS) {
                img = exhip_divide(own_pix, per_image, p.image_magic, p.image_shift);
                in_image = own_pix - img * per_image;
            }
            if (p.residual && own_pix < p.pixels) {
                unsigned from = own_pix;
                if (p.res_shift) {
                    const unsigned oy = exhip_divide(in_image, (unsigned)p.out_w, p.width_magic, p.width_shift), ox = in_image - oy * (unsigned)p.out_w;
                    from = (img * ((unsigned)p.out_h >> p.res_shift) + (oy >> p.res_shift)) * ((unsigned)p.out_w >> p.res_shift) + (ox >> p.res_shift);
                }
                const float* const src = p.residual + (size_t)from * (unsigned)p.rstride + own_ch;
#pragma unroll
                for (int e = 0; e < V; e += 4) {
                    if (p.vector_rows) {
                        if (own_ch + e < p.K) {
                            const v4f r = *reinterpret_cast<const v4f*>(src + e);
#pragma unroll
                            for (int i = 0; i < 4; ++i) res[e + i] = r[i];
                        }
                    } else {
#pragma unroll
                        for (int i = 0; i < 4; ++i) res[e + i] = own_ch + e + i < p.K ? src[e + i] : 0.f;
                    }
                }
            }
        }
        char* const red = lds_all + (wave - part) * BLOCKS * 4096 + lane * 16;
#pragma unroll
        for (int i = 0; i < 4 * BLOCKS; ++i) {
            const v16f& c = acc[i / 4 % MT][i / 4 / MT];
            *reinterpret_cast<v4f*>(red + (part * 4 * BLOCKS + i) * 1024) = v4f{c[i % 4 * 4], c[i % 4 * 4 + 1], c[i % 4 * 4 + 2], c[i % 4 * 4 + 3]};
        }
        __syncthreads();
        if (!owner) return;
#pragma unroll
        for (int j = 0; j < QUADS; ++j) {
            v4f sum = *reinterpret_cast<const v4f*>(red + (quad + j) * 1024);
#pragma unroll
            for (int w = 1; w < WK; ++w) {
                const v4f o = *reinterpret_cast<const v4f*>(red + (w * 4 * BLOCKS + quad + j) * 1024);
#pragma unroll
                for (int e = 0; e < 4; ++e) sum[e] += o[e];
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) v[j * 4 + e] = sum[e];
        }
        if constexpr (ROWS) {
            v16f sum;
#pragma unroll
            for (int e = 0; e < 16; ++e) sum[e] = v[e];
            epilogue_block<MT, SLOW>(p, sum, (tile * NT + quad / 4 / MT) * 32, kb0 + quad / 4 % MT, quad / 4 % MT, lane, lds);
        } else {
            epilogue_part<V>(p, v, par, res, own_pix, img, in_image, own_ch);
        }
    }
}

template <int MT, int NT, int WK, int R, int MODE, bool PAIRS, bool SLOW>
__global__ __launch_bounds__(WK > 4 ? 64 * WK : 256, 2) void conv_f32_kernel(const F32Params p) {
    exhip_touch_args(p);
    __shared__ __attribute__((aligned(16))) char lds_all[F32Shape<MT, NT, WK>::LDS];
    f32_group<MT, NT, WK, R, MODE, PAIRS, SLOW>(p, lds_all, blockIdx.x, gridDim.x);
}

// Two pointwise layers that do not read each other's results in one launch, each in its own form, as conv_pw_two_kernel (conv_pw.hip): a layer
// of a few hundred groups is bounded by its chain of loads and by the gap to the next launch, and two of them fill each other's. The forms are
// those that a detector's neighbours take; any other runs by itself. The layers' parameters are arguments of their own: chosen from an array
// by number they were copied to scratch (792 bytes per lane, 28 - 50 us a launch). Two launches and one, us: 64 and 128 -> 64 channels at
// 1 x 80 x 80 9.7 -> 6.4, at 3 x 80 x 80 14.6 -> 12.2, at 8 x 80 x 80 28.0 -> 27.1; 256 and 512 -> 256 at 1 x 20 x 20 10.1 -> 6.0, at 3
// 13.9 -> 10.6, at 8 21.1 -> 17.4.
struct F32Two {
    int kind[2];
    unsigned groups[2];
};
// the forms by number, -1 for all others
template <int MT, int NT, int WK, int R, int MODE, bool PAIRS, bool SLOW>
constexpr int two_kind() {
    if (MODE != 0 || !PAIRS || SLOW || NT != 1 || R != 8) return -1;
    return MT == 2 ? (WK == 1 ? 0 : WK == 2 ? 1 : WK == 4 ? 2 : -1) : WK == 2 ? 3 : WK == 4 ? 4 : -1;
}
constexpr int kTwoLds = F32Shape<2, 1, 2>::LDS;
__device__ __forceinline__ void two_group(const F32Params& p, int kind, char* lds, unsigned bid, unsigned groups) {
    exhip_touch_args(p);
    if (kind == 0) f32_group<2, 1, 1, 8, 0, true, false>(p, lds, bid, groups);
    else if (kind == 1) f32_group<2, 1, 2, 8, 0, true, false>(p, lds, bid, groups);
    else if (kind == 2) f32_group<2, 1, 4, 8, 0, true, false>(p, lds, bid, groups);
    else if (kind == 3) f32_group<1, 1, 2, 8, 0, true, false>(p, lds, bid, groups);
    else f32_group<1, 1, 4, 8, 0, true, false>(p, lds, bid, groups);
}
__global__ __launch_bounds__(256, 2) void conv_f32_two_kernel(const F32Params a, const F32Params b, const F32Two q) {
    static_assert(F32Shape<2, 1, 1>::LDS <= kTwoLds && F32Shape<2, 1, 4>::LDS <= kTwoLds && F32Shape<1, 1, 2>::LDS <= kTwoLds && F32Shape<1, 1, 4>::LDS <= kTwoLds, "one LDS for all");
    __shared__ __attribute__((aligned(16))) char lds[kTwoLds];
    const unsigned first = q.groups[0];
    if (blockIdx.x < first) two_group(a, q.kind[0], lds, blockIdx.x, first);
    else two_group(b, q.kind[1], lds, blockIdx.x - first, q.groups[1]);
}

thread_local exhip_waiting<F32Params>* t_collect = nullptr;  // (exhip_conv2d_f32_pair)

template <int MT, int NT, int WK, int R, int MODE, bool PAIRS, bool SLOW>
int go(exhip_ctx* ctx, F32Params& p, int kblocks) {
    const long long tiles = ((long long)p.pixels + 32 * NT - 1) / (32 * NT);
    const long long groups = (kblocks + MT - 1) / MT, items = tiles * groups;
    EXHIP_REQUIRE(items < (1ll << 31) - 4, "conv: grid too large");
    p.items = (unsigned)items;
    // Weights that an XCD's 4 MiB of cache do not hold, and that are more than the pixels, are dealt out over the XCDs (512 -> 512
    // 3x3 on one 20 x 20 map, 9.4 MB: 27.5 -> 24.9 us); smaller ones are as fast or faster the other way (2.4 MB: 22.5 against 22.7).
    p.tiles_fast = p.w_bytes > (4u << 20) && p.w_bytes > p.x_bytes;
    p.fast = (unsigned)(p.tiles_fast ? tiles : groups);
    exhip_host_divisor(p.fast, &p.fast_magic, &p.fast_shift);
    const int taps_w = MODE == kPair ? (p.kw + 1) / 2 : p.kw;
    for (int i = 0; i <= WK; ++i) {
        const int s = PAIRS ? (int)((long long)(p.n_ksteps / 2) * i / WK) * 2 : (int)((long long)p.n_ksteps * i / WK), tap = s / p.csteps;
        p.start_s[i] = s;
        p.start_c[i] = s % p.csteps;
        p.start_r[i] = tap / taps_w;
        p.start_q[i] = tap % taps_w * (MODE == kPair ? 2 : 1);
    }
    constexpr int WAVES = F32Shape<MT, NT, WK>::WAVES, ITEMS = F32Shape<MT, NT, WK>::ITEMS;
    if constexpr (two_kind<MT, NT, WK, R, MODE, PAIRS, SLOW>() >= 0) {
        if (t_collect) {
            t_collect->kind = two_kind<MT, NT, WK, R, MODE, PAIRS, SLOW>();
            t_collect->groups = (p.items + ITEMS - 1) / ITEMS;
            t_collect->kernel = reinterpret_cast<const void*>(conv_f32_kernel<MT, NT, WK, R, MODE, PAIRS, SLOW>);
            t_collect->p = p;
            t_collect = nullptr;
            return 0;
        }
    }
    hipLaunchKernelGGL((conv_f32_kernel<MT, NT, WK, R, MODE, PAIRS, SLOW>), dim3((p.items + ITEMS - 1) / ITEMS), dim3(64 * WAVES), 0, ctx->stream, p);
    EXHIP_LAUNCH_CHECK();
    return 0;
}

template <int MODE, bool PAIRS>
int pick(exhip_ctx* ctx, F32Params& p, int kblocks) {
    if (p.act == 4 || p.act == 5) return go<1, 1, 1, 8, MODE, PAIRS, true>(ctx, p, kblocks);
    // The tile and the split that a model of the launch says are shortest, in microseconds: rounds of groups on 256 CUs, each
    // as long as its waves' products (0.028 a product and SIMD), the blocks' epilogue (1 each, shared by the waves of a tile) and
    // the exchange of a split (0.4), or the time the operands take at 12 TB/s where that is longer. Over 28 layers from
    // 1 x 64 x 8 x 4 to 30 GFLOP its choice is within 1 % of the fastest form of the list on average.
    struct Config { int mt, nt, wk; };
    static constexpr Config kConfigs[] = {{2, 2, 1}, {2, 1, 1}, {2, 1, 2}, {2, 1, 4}, {1, 1, 4}, {1, 1, 8}, {1, 2, 1}, {1, 1, 2}};
    constexpr int kCount = (int)(sizeof(kConfigs) / sizeof(kConfigs[0]));
    int best = 0;
    double best_cost = 0;
    for (int i = 0; i < kCount; ++i) {
        const Config& c = kConfigs[i];
        if (c.wk > p.n_ksteps) continue;
        const int blocks = c.mt * c.nt, waves = std::max(4, c.wk), steps = (p.n_ksteps + c.wk - 1) / c.wk;
        const double tiles = (double)(((long long)p.pixels + 32 * c.nt - 1) / (32 * c.nt) * ((kblocks + c.mt - 1) / c.mt));
        const double rounds = std::ceil(std::ceil(tiles * c.wk / waves) / 256) * (waves / 4);
        const double round = steps * blocks * 4 * 0.0278 + (double)blocks / std::min(c.wk, blocks) + (c.wk > 1 ? 0.4 : 0);
        const double cost = std::max(rounds * round, tiles * c.wk * steps * (c.mt + c.nt) * 1024 / 12e6);
        if (i == 0 || cost < best_cost) {
            best_cost = cost;
            best = i;
        }
    }
    if (g_exhip_options.f32_tile > 0) best = std::min(g_exhip_options.f32_tile, kCount) - 1;
    switch (best) {
    case 0: return go<2, 2, 1, 4, MODE, PAIRS, false>(ctx, p, kblocks);
    case 1: return go<2, 1, 1, PAIRS ? 8 : 6, MODE, PAIRS, false>(ctx, p, kblocks);
    case 2: return go<2, 1, 2, PAIRS ? 8 : 6, MODE, PAIRS, false>(ctx, p, kblocks);
    case 3: return go<2, 1, 4, PAIRS ? 8 : 6, MODE, PAIRS, false>(ctx, p, kblocks);
    case 4: return go<1, 1, 4, 8, MODE, PAIRS, false>(ctx, p, kblocks);
    case 5: return go<1, 1, 8, 8, MODE, PAIRS, false>(ctx, p, kblocks);
    case 6: return go<1, 2, 1, PAIRS ? 8 : 6, MODE, PAIRS, false>(ctx, p, kblocks);
    default: return go<1, 1, 2, 8, MODE, PAIRS, false>(ctx, p, kblocks);
    }
}

int taps_steps(const exhip_conv_desc* d) { return d->c_stride == 4 ? d->kh * ((d->kw + 1) / 2) : d->kh * d->kw * ((d->c + 7) / 8); }

}  // namespace

int exhip_conv_f32_validate(const exhip_conv_desc* d) {
    EXHIP_REQUIRE(d, "conv: NULL descriptor");
    EXHIP_REQUIRE(d->n > 0 && d->c > 0 && d->h > 0 && d->w > 0 && d->k > 0, "conv: empty shape");
    EXHIP_REQUIRE(d->kh > 0 && d->kw > 0 && d->sh > 0 && d->sw > 0, "conv: bad kernel/stride");
    EXHIP_REQUIRE(d->sh == d->sw, "conv: MFMA path needs equal strides (got %dx%d)", d->sh, d->sw);
    EXHIP_REQUIRE(d->pt >= 0 && d->pb >= 0 && d->pl >= 0 && d->pr >= 0, "conv: negative padding");
    EXHIP_REQUIRE(d->h + d->pt + d->pb >= d->kh && d->w + d->pl + d->pr >= d->kw, "conv: kernel larger than padded input");
    EXHIP_REQUIRE(d->c_stride >= d->c, "conv: c_stride %d < c %d", d->c_stride, d->c);
    EXHIP_REQUIRE(d->c_stride == 4 || d->c_stride % 8 == 0, "conv: input pixel is %d bytes; need a multiple of 32, or 16", d->c_stride * 4);
    EXHIP_REQUIRE((long long)d->h * d->w * d->c_stride * 4 < (1ll << 31), "conv: one input image exceeds 2 GiB");
    EXHIP_REQUIRE((long long)((d->k + 31) / 32) * taps_steps(d) * 1024 < (1ll << 31), "conv: the packed weights exceed 2 GiB");
    return 0;
}

size_t exhip_conv_f32_packed_bytes(const exhip_conv_desc* d) {
    if (exhip_conv_f32_validate(d)) return 0;
    if (exhip_conv_f32_thirds(d)) return exhip_conv_f32_thirds_bytes(d);
    return (size_t)((d->k + 31) / 32) * taps_steps(d) * 1024;
}

// [32-channel block][step: filter row, tap, 8 channels (or 2 taps x 4 channels)][lane][4 floats]; the accumulator of
// v_mfma_f32_32x32x2_f32 then holds sixteen neighbouring channels per lane.
int exhip_conv_f32_pack_weights(const exhip_conv_desc* d, const float* w, float* out) {
    const int rc = exhip_conv_f32_validate(d);
    if (rc) return rc;
    if (exhip_conv_f32_thirds(d)) {
        exhip_conv_f32_thirds_pack(d, w, out);
        return 0;
    }
    const bool pair = d->c_stride == 4;
    const int C = d->c, K = d->k, KH = d->kh, KW = d->kw, csteps = pair ? 1 : (C + 7) / 8;
    const int taps_w = pair ? (KW + 1) / 2 : KW;
    const size_t tap_step = (size_t)csteps * 256;  // floats from a tap's vectors to the next one's
    for (int kb = 0; kb < (K + 31) / 32; ++kb, out += KH * taps_w * tap_step) {
        auto channel = [kb](int rr) { return kb * 32 + ((rr / 4) % 2) * 16 + (rr / 8) * 4 + rr % 4; };
        if (pair) {
            for (int lane = 0; lane < 64; ++lane)
                for (int r = 0; r < KH; ++r)
                    for (int q = 0; q < taps_w; ++q)
                        for (int e = 0; e < 4; ++e) {
                            const int k = channel(lane % 32), tap = 2 * q + lane / 32;
                            out[(r * taps_w + q) * tap_step + lane * 4 + e] = k < K && e < C && tap < KW ? w[(((size_t)k * C + e) * KH + r) * KW + tap] : 0.f;
                        }
            continue;
        }
        for (int j = 0; j < csteps; ++j)
            exhip_pack_block<float>(
                [&](int rr, int half, int* n) {
                    const int k = channel(rr), c = j * 8 + half * 4;
                    *n = k < K ? std::max(0, std::min(4, C - c)) : 0;
                    return *n ? w + ((size_t)k * C + c) * KH * KW : w;
                },
                KH * KW, reinterpret_cast<char*>(out + j * 256), tap_step * 4);
    }
    return 0;
}

static int run_conv_f32(exhip_ctx* ctx, const exhip_conv_desc* d, const exhip_conv_place* place, const float* x, const void* wp, const float* bias,
                        const float* residual, float* y, float* y_nchw) {
    EXHIP_REQUIRE(y || y_nchw, "exhip_conv2d_f32: no output requested");
    EXHIP_REQUIRE(ctx, "conv: NULL ctx");
    const int rc = exhip_conv_f32_validate(d);
    if (rc) return rc;
    if (!place && (d->post_bn_a || d->post_bn_b || d->exact_k)) return EXHIP_ERR_UNSUPPORTED;  // the placed entry's
    EXHIP_REQUIRE(x && wp, "conv: NULL input or weights");
    const int layout = place ? place->layout : EXHIP_PLACE_ROWS, group = place ? place->group : 0;
    EXHIP_REQUIRE(layout != EXHIP_PLACE_ROWS || d->k_stride >= d->k || (!y && !residual), "conv: k_stride %d < k %d", d->k_stride, d->k);
    EXHIP_REQUIRE(!bias || (uintptr_t)bias % 16 == 0, "conv: scale and bias arrays must be 16-byte aligned");
    EXHIP_REQUIRE((uintptr_t)x % 16 == 0 && (uintptr_t)wp % 16 == 0, "conv: input and weights must be 16-byte aligned");
    EXHIP_REQUIRE((d->post_op >= 0 && d->post_op <= 1 + EXHIP_UNARY_CLIP && d->post_op != 1 + EXHIP_UNARY_SIGMOID) ||
                      (d->post_op == EXHIP_POST_PRELU && d->post_slope),
                  "conv: post_op %d is not an activation the epilogue applies", d->post_op);
    EXHIP_REQUIRE((d->post_bn_a == nullptr) == (d->post_bn_b == nullptr), "conv: half a BatchNorm");
    F32Params p = {};
    const int oh = (d->h + d->pt + d->pb - d->kh) / d->sh + 1, ow = (d->w + d->pl + d->pr - d->kw) / d->sw + 1;
    p.layout = layout;
    p.group = group;
    p.rstride = d->k_stride;
    if (place) {
        EXHIP_REQUIRE(layout >= EXHIP_PLACE_ROWS && layout <= EXHIP_PLACE_SHUFFLED && place->residual_shift >= 0 && place->residual_shift <= 4,
                      "conv: unknown placement");
        EXHIP_REQUIRE(layout == EXHIP_PLACE_ROWS || (group > 0 && d->k % group == 0 && y && !y_nchw), "conv: %d channels do not make groups of %d", d->k, group);
        EXHIP_REQUIRE(layout != EXHIP_PLACE_SHUFFLED || (d->k == 4 * group && d->k_stride >= group), "conv: a shuffled layer has four groups");
        EXHIP_REQUIRE(!residual || (place->residual_stride >= d->k && oh % (1 << place->residual_shift) == 0 && ow % (1 << place->residual_shift) == 0),
                      "conv: the shortcut does not fit the output");
        p.rstride = place->residual_stride;
        p.res_shift = residual ? place->residual_shift : 0;
        p.bn_relu = place->bn_relu;
    }
    p.wp = static_cast<const char*>(wp);
    p.bias = bias; p.bn_a = d->post_bn_a; p.bn_b = d->post_bn_b;
    p.slope = d->post_op == EXHIP_POST_PRELU ? d->post_slope : nullptr;
    p.in_h = d->h; p.in_w = d->w; p.out_h = oh; p.out_w = ow;
    p.stride = d->sh; p.pad_t = d->pt; p.pad_l = d->pl; p.kh = d->kh; p.kw = d->kw;
    p.xs_b = d->c_stride * 4;
    p.row_b = d->w * p.xs_b;
    const bool pair = d->c_stride == 4;
    const bool thirds = exhip_conv_f32_thirds(d);
    p.csteps = thirds ? d->c / 16 : pair ? 1 : (d->c + 7) / 8;
    p.n_ksteps = taps_steps(d);
    p.w_bytes = (unsigned)(thirds ? exhip_conv_f32_thirds_bytes(d) : (size_t)((d->k + 31) / 32) * p.n_ksteps * 1024);
    p.K = d->k;
    p.kstride = d->k_stride;
    p.k_end = d->exact_k || !y || layout != EXHIP_PLACE_ROWS ? d->k : std::max(d->k, d->k_stride);
    p.act = d->act; p.post_relu = d->post_relu; p.post_op = d->post_op; p.slope_shared = d->post_slope_shared;
    p.residual_last = d->residual_last;
    p.alpha = d->post_alpha; p.beta = d->post_beta;
    p.vector_rows = d->k_stride % 4 == 0 && (uintptr_t)y % 16 == 0 && p.k_end % 4 == 0 &&
                    (!residual || ((uintptr_t)residual % 16 == 0 && p.rstride % 4 == 0 && (d->k + 3) / 4 * 4 <= p.rstride));
    if (layout == EXHIP_PLACE_SHUFFLED && group % 32 != 0) p.vector_rows = 0;
    exhip_host_divisor((unsigned)(oh * ow), &p.image_magic, &p.image_shift);
    exhip_host_divisor((unsigned)ow, &p.width_magic, &p.width_shift);
    // blocks past the last channel's (pad channels of a wider stride) get zeros too: weights beyond the view read zero
    const int write_blocks = (p.k_end + 31) / 32;
    const long long img_bytes = (long long)d->h * p.row_b, per_image = (long long)oh * ow;
    EXHIP_REQUIRE(per_image < (1ll << 29) && (layout != EXHIP_PLACE_GROUPED || per_image * d->k < (1ll << 31)), "conv: too many output pixels in an image");
    // input offsets are 32-bit, pixel numbers 31-bit, offsets of grouped results 32-bit: as many images per launch as fit
    long long most = std::min(0x7fff0000ll / img_bytes, ((1ll << (thirds || layout == EXHIP_PLACE_SHUFFLED ? 29 : 31)) - 256) / per_image);
    if (layout == EXHIP_PLACE_GROUPED) most = std::min(most, (1ll << 32) / (per_image * d->k) - 1);
    most = std::max(1ll, most);
    const long long y_image = layout == EXHIP_PLACE_SHUFFLED ? per_image * 4 * d->k_stride : layout == EXHIP_PLACE_GROUPED ? per_image * d->k : per_image * d->k_stride;
    for (long long n0 = 0; n0 < d->n; n0 += most) {
        const long long n = std::min<long long>(most, d->n - n0);
        p.x = reinterpret_cast<const char*>(x) + n0 * img_bytes;
        p.x_bytes = (unsigned)(n * img_bytes);
        p.pixels = (unsigned)(n * per_image);
        p.residual = residual ? residual + n0 * (per_image >> (2 * p.res_shift)) * p.rstride : nullptr;
        p.y = y ? y + n0 * y_image : nullptr;
        p.y_nchw = y_nchw ? y_nchw + n0 * per_image * d->k : nullptr;
        // 1x1 layers of whole 64-byte pieces take the pixels in pairs of steps: 512 -> 256 on one 20 x 20 map 6.05 -> 5.44 us, 1024 -> 512 on
        // three 13 x 13 maps 9.1 -> 8.3. With a filter the products bound the chain, and the detour through LDS only lengthens it
        // (64 -> 64 3x3 on one 160 x 160 map 23.6 us, 25.2 in pairs, 18.8 in thirds).
        const bool point = d->kh == 1 && d->kw == 1 && !d->pt && !d->pb && !d->pl && !d->pr;
        const int go_rc = thirds                ? exhip_conv_f32_thirds_run(ctx, {&p, n, write_blocks})
                          : pair                  ? pick<kPair, false>(ctx, p, write_blocks)
                          : !point              ? pick<kTaps, false>(ctx, p, write_blocks)
                          : p.csteps % 2 == 0   ? pick<kPoint, true>(ctx, p, write_blocks)
                                                : pick<kPoint, false>(ctx, p, write_blocks);
        if (go_rc) return go_rc;
    }
    return 0;
}

extern "C" int exhip_conv2d_f32(exhip_ctx* ctx, const exhip_conv_desc* d, const float* x, const void* wp,
                                const float* bias, const float* residual, float* y_f32_nhwc, float* y_f32_nchw) {
    return run_conv_f32(ctx, d, nullptr, x, wp, bias, residual, y_f32_nhwc, y_f32_nchw);
}

extern "C" int exhip_conv2d_f32_placed(exhip_ctx* ctx, const exhip_conv_desc* d, const exhip_conv_place* place, const float* x, const void* wp,
                                       const float* bias, const float* residual, float* y, float* y_f32_nchw) {
    EXHIP_REQUIRE(place, "exhip_conv2d_f32_placed: NULL placement");
    return run_conv_f32(ctx, d, place, x, wp, bias, residual, y, y_f32_nchw);
}

extern "C" int exhip_conv2d_f32_pair(exhip_ctx* ctx, const exhip_conv_f32_call* a, const exhip_conv_f32_call* b) {
    EXHIP_REQUIRE(ctx && a && b && a->d && a->place && b->d && b->place, "exhip_conv2d_f32_pair: NULL argument");
    auto layer = [](exhip_ctx* on, const void* call) {
        const auto* c = static_cast<const exhip_conv_f32_call*>(call);
        return exhip_conv2d_f32_placed(on, c->d, c->place, c->x, c->w_packed, c->bias, c->residual, c->y, c->y_nchw);
    };
    return exhip_run_pair(ctx, &t_collect, layer, a, b, [ctx](const exhip_waiting<F32Params>* w) {
        const F32Two q = {{w[0].kind, w[1].kind}, {w[0].groups, w[1].groups}};
        hipLaunchKernelGGL(conv_f32_two_kernel, dim3(w[0].groups + w[1].groups), dim3(256), 0, ctx->stream, w[0].p, w[1].p, q);
        EXHIP_LAUNCH_CHECK();
        return 0;
    });
}
