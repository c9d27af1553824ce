// What the kernels for fp16 and int8 NHWC convolutions without a plan of tiles share (conv_pw.hip, conv_staged.hip): a launch's parameters, the layers
// behind the products, and how results reach memory.
#pragma once
#include <hip/hip_runtime.h>

#include <cfloat>
#include <cstdint>
#include <type_traits>

#include "conv_pw.h"
#include "pw_rows.h"

namespace {

typedef exhip_v4i v4i;
typedef float v16f __attribute__((ext_vector_type(16)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

constexpr unsigned kRsrcWord3 = 0x00020000u;  // raw buffer: out-of-range loads return 0
constexpr int kOutOfRange = kPwOutOfRange;    // a lane offset beyond every view
constexpr int kMaxDirectSteps = 40;           // table entries of a layer with a filter, a k-step (taps x 32-byte steps per pixel) or a pair each
constexpr int kSplit = 4;                     // waves that share a tile's k-steps in the split form
constexpr int kTapShift = 27;                 // a step's table entry: byte offset below, tap number above

struct PwParams {
    const char* x;
    const char* wp;
    const float* bias;
    const uint16_t* residual;
    uint16_t* y;
    const float* post_slope;
    // int8 layers: dequantization scales, float32 shortcut, float32 and int8 results
    const float* scale;
    const float* residual_f;
    float* y_f;
    int8_t* y_q;
    float fs_out;
    const float* post_bn_a;   // BatchNorm in front of post_op: fmaf(post_bn_b[ch], v, post_bn_a[ch])
    const float* post_bn_b;
    int group;                // a detection head: results go to [image][channel / group][pixel][channel % group] (0: rows)
    int exact;                // channels [0, K) only: blocks past K are not written (the results lie inside a wider tensor)
    unsigned pixels, x_bytes, w_bytes;
    unsigned items, ch_groups;   // waves with work; 32 * MT channel groups per pixel tile
    unsigned groups_magic, image_magic, width_magic;  // exhip_divide() by ch_groups, out_h * out_w, out_w
    int groups_shift, image_shift, width_shift;
    int xs_b;                    // bytes per input pixel
    int n_ksteps;                // 32-byte k-steps per pixel
    int mts;                     // 32-channel blocks per packed slab
    int K, kstride;
    int act, post_relu, post_op, post_slope_shared, residual_last;
    float post_alpha, post_beta;
    // the form with a filter (TAPS): output pixel (img, oy, ox) reads input pixel (oy * stride - pt + r, ox * stride - pl + q)
    // for k-step s of tap r * kw + q, that many bytes behind its top-left input pixel
    int in_h, in_w, out_h, out_w, stride, pad_t, pad_l, kh, kw;
    int step[kMaxDirectSteps];   // of a k-step or pair: offset | tap << kTapShift (not used by the split form)
    int pair_first[kMaxDirectSteps];  // the weights' k-step of a pair's first
    // the split form: where each wave of a tile begins -- its first k-step (and that of its weights), bytes behind the top-left input pixel,
    // filter row, tap and bytes left of the chunk -- and what leads from behind a row's last tap to the next row, and from
    // behind the last row to the next chunk
    int start_s[kSplit + 1], start_w[kSplit + 1], start_b[kSplit + 1], start_r[kSplit + 1], start_q[kSplit + 1], start_left[kSplit + 1];
    int chunk_b, row_end_b, chunk_end_b, pool;
    int pair_w, next_w, chunk_w;  // pairs: k-steps of the weights from a pair's first to its second, to the next pair, and more behind the last tap
    // the depthwise 3x3 layer in front (dw_pw_kernel; geometry in in_h .. pad_l above, x is its input): weights, bias and PReLU slopes,
    // activation 0, 1 or 3; 32-pixel tiles of a group and output blocks of a group
    const float* dw_w;
    const float* dw_bias;
    const float* dw_slope;
    int dw_act, dw_slope_shared, dw_pixels, dw_tiles, dw_kblocks, dw_split, dw_mid, kblocks;  // dw_mid: where its results begin in LDS
    // the first layer on NCHW planes (stem_planes_kernel; geometry in in_h .. pad_l above, x is its input): channels, the Input layer's means and
    // factors (or NULL), output rows of a group, groups an image (ch_groups), pixels of a row in LDS, 16-byte pieces of an input row
    const float* mean;
    const float* factor;
    float fs_in;  // the quantizer's
    int in_c, tile_rows, row_pixels, pieces, pieces_shift;
    unsigned pieces_magic;
};

__device__ __noinline__ float slow_activation(float v, int act) { return exhip_act(v, act); }

// ---- epilogue ----
// What bounds a short launch is the length of one wave's chain, and the epilogue was half of it (stamps inside a 256 -> 256
// layer on a 20 x 20 map, 19 000 cycles in all: 3 000 for 32 conditional one-word bias loads, 4 200 - 8 200 for the arithmetic
// with a test per value, per lane and per layer kind, most of it instruction fetch, against 7 000 for the products). So:
//  * the per-channel parameters (scale, bias, BatchNorm, PReLU slopes) are requested at the kernel's start, one coalesced
//    load each with zeros beyond K, wait in the wave's own LDS slice and are read back four channels at a time;
//  * the layers behind the convolution are template constants (Ep) for the combinations the networks are made of, so the
//    epilogue is straight code; any other combination runs the one instantiation that looks at run time (Any);
//  * results leave through the LDS slice, so that every store instruction writes whole rows of MT * 32 channels.
enum { kPostNone, kPostRelu, kPostHardSwish, kPostLeaky, kPostPrelu, kPostHardSigmoid, kPostClip };
template <int ACT, int POST, int RES, bool BN, bool ANY>
struct EpT {
    static constexpr int act = ACT, post = POST, res = RES;  // res: 0 no shortcut, 1 added in front of the layers behind, 2 behind them
    static constexpr bool bn = BN, any = ANY, pool = false;
};
// ... and a 2x2 stride-2 max pooling of whole windows behind them all: four neighbouring lanes have a window's pixels (p.out_h, p.out_w: the pooled map).
// Spares a large layer the float32 map, which is most of its bytes: 32 -> 32 at 64 x 126 x 126 39.6 us and 28.1 for the pooling -> 32.3.
template <typename E>
struct Pooled : E {
    static constexpr bool pool = true;
};
template <int ACT, int POST, int RES, bool BN = false>
using Ep = EpT<ACT, POST, RES, BN, false>;
using EpAny = EpT<0, 0, 0, false, true>;

constexpr int kParams = 4;  // scale / bias / BatchNorm a or PReLU slope / BatchNorm b
constexpr int param_bytes(int mt) { return kParams * mt * 32 * 4; }
constexpr int tile_bytes(int dt, int mt) { return 32 * ((dt == EXHIP_I8 ? 128 : mt * 64) + 16); }  // int8 layers: one float32 block
constexpr int wave_bytes(int dt, int mt) { return param_bytes(mt) + tile_bytes(dt, mt); }

// N neighbouring channels' parameters from channel `at` of the wave's MT * 32 on.
template <int MT, int N>
__device__ __forceinline__ void read_parameters(const char* lds, int which, int at, float (&v)[N]) {
    const v4f* src = reinterpret_cast<const v4f*>(lds + (which * MT * 32 + at) * 4);
#pragma unroll
    for (int q = 0; q < N / 4; ++q) {
        const v4f t = src[q];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[q * 4 + e] = t[e];
    }
}

// ROUND: the layer behind reads the halves that the layer in front of it stored.
template <bool ROUND, int N>
__device__ __forceinline__ void stored(float (&v)[N]) {
    if constexpr (ROUND) {
#pragma unroll
        for (int e = 0; e < N; e += 2) {
            const unsigned d = exhip_round_pair(v[e], v[e + 1]);
            v[e] = exhip_h2f((uint16_t)(d & 0xffff));
            v[e + 1] = exhip_h2f((uint16_t)(d >> 16));
        }
    }
}

template <int OP, bool ROUND, int N>
__device__ __forceinline__ void unary_values(float (&v)[N], float alpha, float beta) {
    stored<ROUND>(v);
#pragma unroll
    for (int e = 0; e < N; ++e) v[e] = unary_value<OP>(v[e], alpha, beta);
}

template <bool ROUND, int N>
__device__ __forceinline__ void relu_values(float (&v)[N]) {
    stored<ROUND>(v);
#pragma unroll
    for (int e = 0; e < N; ++e) v[e] = (0.f > v[e]) ? 0.f : v[e];
}

// Rows of a wave tile from its LDS slice to memory: CHUNKS 16-byte pieces per row of 32, neighbouring lanes on neighbouring
// pieces. The view starts at the tile's first pixel and channel and ends behind its last pixel's row; `bytes`: how far the
// tensor's channels reach from the tile's first one.
template <int CHUNKS>
__device__ __forceinline__ void store_rows(const char* tile, int pitch, __amdgpu_buffer_rsrc_t y, int row_bytes, int bytes, int lane) {
    const int row = lane / CHUNKS, col = (lane % CHUNKS) * 16;
    const int at = pw_lane_offset(row, row_bytes, col, bytes);
#pragma unroll
    for (int j = 0; j < CHUNKS / 2; ++j) {
        const v4i t = *reinterpret_cast<const v4i*>(tile + (j * (64 / CHUNKS) + row) * pitch + col);
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(__attribute__((ext_vector_type(4))) unsigned int, t), y, at, j * (64 / CHUNKS) * row_bytes, 0);
    }
}

// A view of a pixel-major tensor from pixel `first` and channel ch0 on, `rows` pixels long.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t tile_view(const void* base, unsigned first, int row_bytes, int ch_bytes, int rows) {
    char* p = const_cast<char*>(static_cast<const char*>(base)) + (size_t)first * (unsigned)row_bytes + ch_bytes;
    return __builtin_amdgcn_make_buffer_rsrc(p, 0, pw_view_bytes(rows, row_bytes, ch_bytes), kRsrcWord3);
}

// The layers behind the products and the bias, of N neighbouring channels from channel `at` of the wave's MT * 32 on; residual(e): the
// shortcut's value. (An activation that only EpAny has is evaluated value by value, so that its registers are needed once.)
template <int DT, int MT, typename EP, int N, typename RES>
__device__ __forceinline__ void layers_behind(const PwParams& p, float (&v)[N], const char* lds, int at, bool shortcut, RES residual) {
    constexpr bool I8 = DT == EXHIP_I8, ANY = EP::any;
    float t[N];
    if (ANY ? p.act == 1 : EP::act == 1) relu_values<false>(v);
    if (ANY && p.act > 1) {
#pragma unroll 1
        for (int e = 0; e < N; ++e) v[e] = slow_activation(v[e], p.act);
    }
    auto add_shortcut = [&]() {
        stored<!I8>(v);
#pragma unroll
        for (int e = 0; e < N; ++e) v[e] += residual(e);
    };
    if (ANY ? shortcut && !p.residual_last : EP::res == 1) add_shortcut();
    if (ANY ? p.post_relu != 0 : EP::post == kPostRelu) relu_values<!I8>(v);
    if (I8 && (ANY ? p.post_bn_a != nullptr : EP::bn)) {  // the BatchNorm layer between this layer (through a Concat) and its activation layer
        float a[N], b[N];
        read_parameters<MT>(lds, 2, at, a);
        read_parameters<MT>(lds, 3, at, b);
#pragma unroll
        for (int e = 0; e < N; ++e) v[e] = __builtin_fmaf(b[e], v[e], a[e]);
    }
    if (ANY ? p.post_op == 1 + EXHIP_UNARY_HARDSWISH : EP::post == kPostHardSwish) unary_values<0, !I8>(v, p.post_alpha, p.post_beta);
    if (ANY ? p.post_op == 1 + EXHIP_UNARY_LEAKYRELU : EP::post == kPostLeaky) unary_values<1, !I8>(v, p.post_alpha, p.post_beta);
    if (ANY && p.post_op == 1 + EXHIP_UNARY_HARDSIGMOID) unary_values<3, !I8>(v, p.post_alpha, p.post_beta);
    if (ANY && p.post_op == 1 + EXHIP_UNARY_CLIP) unary_values<4, !I8>(v, p.post_alpha, p.post_beta);
    if (ANY ? p.post_op == EXHIP_POST_PRELU : EP::post == kPostPrelu) {
        read_parameters<MT>(lds, 2, at, t);
        stored<!I8>(v);
#pragma unroll
        for (int e = 0; e < N; ++e) v[e] = v[e] >= 0.f ? v[e] : t[e] * v[e];
    }
    if (ANY ? shortcut && p.residual_last : EP::res == 2) add_shortcut();
}

template <int DT, int MT, int NT, typename EP, typename ACC>
__device__ __forceinline__ void pw_epilogue(const PwParams& p, const ACC (&acc)[MT][NT], unsigned pix0, unsigned end, int kb0, int lane, char* lds) {
    constexpr bool I8 = DT == EXHIP_I8, ANY = EP::any;
    constexpr int ES = I8 ? 4 : 2;  // bytes per value of the shortcut tensor
    const int half = lane >> 5, row = lane & 31;
    char* const tile = lds + param_bytes(MT);
    const int k_end = pw_channel_end(p.K, p.kstride, p.exact);
    const bool shortcut = ANY ? (I8 ? p.residual_f != nullptr : p.residual != nullptr) : EP::res != 0;
    // grouped results: every half-wave writes the 32 channels of one pixel of a block, runs of neighbouring values (a head of 128 -> 255
    // channels at 16 x 80 x 80 takes 37 us, the memory's time for its 104 MB is 20; without this form, 41 us and a second launch over them)
    auto store_grouped = [&](auto* y, int pitch, int at0, unsigned first, int rows, int kb) {
        typedef typename std::remove_pointer<decltype(y)>::type T;
        const unsigned per_image = (unsigned)(p.out_h * p.out_w), img = exhip_divide(first + row, per_image, p.image_magic, p.image_shift);
        const unsigned lane_at = img * (unsigned)p.K * per_image + (first + row - img * per_image) * (unsigned)p.group;
        const int ch = kb * 32 + row, g = ch / p.group, member = ch - g * p.group;
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int srow = j * 2 + half;
            const unsigned at = (unsigned)__builtin_amdgcn_ds_bpermute(srow * 4, (int)lane_at) + (unsigned)g * per_image * (unsigned)p.group + member;
            if (srow < rows && ch < p.K) y[at] = *reinterpret_cast<const T*>(tile + srow * pitch + at0 + row * (int)sizeof(T));
        }
    };
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        const unsigned first = pix0 + n * 32;
        if (n > 0 && first >= end) continue;
        const int rows = end - first < 32 ? (int)(end - first) : 32;
        v4i r[MT][ES];
        if (shortcut) {
            // a channel group beyond the tensor's stride reads zeros; pad channels inside it read what lies there and are
            // overwritten with zeros below
            const __amdgpu_buffer_rsrc_t rr = tile_view(I8 ? (const void*)p.residual_f : (const void*)p.residual, first, p.kstride * ES, kb0 * 32 * ES, rows);
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int q = 0; q < ES; ++q) {
                    const int ch = m * 32 + half * 16 + q * (16 / ES);
                    const int at = pw_lane_offset(row, p.kstride * ES, ch * ES, (p.kstride - kb0 * 32) * ES);
                    r[m][q] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rr, at, 0, 0));
                }
        }
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const int kb = kb0 + m, ch0 = kb * 32 + half * 16;
            if (m > 0 && !pw_block_exists(kb, k_end)) continue;
            float v[16], t[16];
            if constexpr (I8) {
                float b[16];
                read_parameters<MT>(lds, 0, m * 32 + half * 16, t);
                read_parameters<MT>(lds, 1, m * 32 + half * 16, b);
#pragma unroll
                for (int e = 0; e < 16; ++e) v[e] = __builtin_fmaf((float)acc[m][n][e], t[e], b[e]);
            } else {
                read_parameters<MT>(lds, 1, m * 32 + half * 16, t);
#pragma unroll
                for (int e = 0; e < 16; ++e) v[e] = acc[m][n][e] + t[e];
            }
            layers_behind<DT, MT, EP>(p, v, lds, m * 32 + half * 16, shortcut, [&](int e) {
                const int word = r[m][I8 ? e >> 2 : e >> 3][I8 ? e & 3 : (e >> 1) & 3];  // (a bit cast of the element itself takes the vector's first)
                if constexpr (I8) return __builtin_bit_cast(float, word);
                else return exhip_h2f((uint16_t)(((uint32_t)word >> ((e & 1) * 16)) & 0xffff));
            });
            if (kb * 32 + 32 > p.K) {  // pad channels hold zeros (wave-uniform: only the block with the ragged end looks)
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    if (ch0 + e >= p.K) v[e] = 0.f;
            }
            if constexpr (EP::pool) {
                // the maximum over the quad's lanes, as the pooling kernel takes it (a NaN never is the larger one); each of them then stores
                // four of the channels
                const int member = lane & 3, ch = half * 16 + member * 4, pixel = row >> 2, quads = rows >> 2;
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    v[e] = -FLT_MAX < v[e] ? v[e] : -FLT_MAX;
                    const float beside = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v[e]), 0xB1, 0xF, 0xF, true));
                    v[e] = v[e] < beside ? beside : v[e];
                    const float below = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v[e]), 0x4E, 0xF, 0xF, true));
                    v[e] = v[e] < below ? below : v[e];
                }
                v4f o;
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = member == 0 ? v[e] : member == 1 ? v[4 + e] : member == 2 ? v[8 + e] : v[12 + e];
                typedef unsigned v4u __attribute__((ext_vector_type(4)));
                if (p.y_f)
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, o), tile_view(p.y_f, first >> 2, p.kstride * 4, kb * 128, quads),
                                                           pw_lane_offset(pixel, p.kstride * 4, ch * 4, (k_end - kb * 32) * 4), 0, 0);
                if (p.y_q) {
                    uint32_t w = 0;
#pragma unroll
                    for (int e = 0; e < 4; ++e) w |= (uint32_t)(exhip_q8(o[e] * p.fs_out) & 0xff) << (8 * e);
                    __builtin_amdgcn_raw_buffer_store_b32(w, tile_view(p.y_q, first >> 2, p.kstride, kb * 32, quads), pw_lane_offset(pixel, p.kstride, ch, k_end - kb * 32), 0, 0);
                }
            } else if constexpr (I8) {
                if (p.y_f) {  // one block at a time: 128 bytes per pixel
                    constexpr int pitch = 128 + 16;
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const v4f o = {v[q * 4], v[q * 4 + 1], v[q * 4 + 2], v[q * 4 + 3]};
                        *reinterpret_cast<v4f*>(tile + row * pitch + half * 64 + q * 16) = o;
                    }
                    if (ANY && p.group) store_grouped(p.y_f, pitch, 0, first, rows, kb);
                    else store_rows<8>(tile, pitch, tile_view(p.y_f, first, p.kstride * 4, kb * 128, rows), p.kstride * 4, (k_end - kb * 32) * 4, lane);
                }
                if (p.y_q) {
                    v4i o;
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        uint32_t w = 0;
#pragma unroll
                        for (int e = 0; e < 4; ++e) w |= (uint32_t)(exhip_q8(v[q * 4 + e] * p.fs_out) & 0xff) << (8 * e);
                        o[q] = (int)w;
                    }
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(__attribute__((ext_vector_type(4))) unsigned int, o),
                                                           tile_view(p.y_q, first, p.kstride, kb * 32, rows),
                                                           pw_lane_offset(row, p.kstride, half * 16, k_end - kb * 32), 0, 0);
                }
            } else {
                constexpr int pitch = MT * 64 + 16;
                v4i o[2];
#pragma unroll
                for (int e = 0; e < 8; ++e) o[e >> 2][e & 3] = (int)exhip_round_pair(v[2 * e], v[2 * e + 1]);
                *reinterpret_cast<v4i*>(tile + row * pitch + m * 64 + half * 32) = o[0];
                *reinterpret_cast<v4i*>(tile + row * pitch + m * 64 + half * 32 + 16) = o[1];
            }
            // one 32 x 32 block at a time: interleaving the blocks buys nothing and costs the registers of their temporaries
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (!I8) {
            if (ANY && p.group) {
#pragma unroll
                for (int m = 0; m < MT; ++m) store_grouped(p.y, MT * 64 + 16, m * 64, first, rows, kb0 + m);
                continue;
            }
        }
        if constexpr (!I8)
            store_rows<MT * 4>(tile, MT * 64 + 16, tile_view(p.y, first, p.kstride * 2, kb0 * 64, rows), p.kstride * 2, (k_end - kb0 * 32) * 2, lane);
    }
}

}  // namespace
