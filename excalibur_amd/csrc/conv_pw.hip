// conv1x1_pw_kernel: the pointwise (1x1, stride 1, no padding) convolution on half or int8 NHWC tensors, y[pixel][k] = sum_c x[pixel][c]
// * w[k][c]; its tapped form (TAPS) for layers with a filter, a stride or padding; conv_pw_split_kernel, several waves to a tile;
// dw_pw_kernel, a depthwise 3x3 layer in front; and stem_planes_kernel, a network's first layer from its planes.
//
// A pointwise layer of a detection or mobile network moves a few tens of MB for a few GFLOP: what it costs is the
// length of one group's chain from launch to last store, and the memory system's rate. So no operand is staged: a wave
// owns 32 * NT pixels x 32 * MT output channels and fetches its MFMA operands straight into registers, 16 bytes per
// lane and k-step -- the weight fragments in the general kernel's packing (one contiguous KiB per 32-channel block and
// k-step), the pixel fragments from the NHWC rows themselves (lane = pixel, the two half-waves the two 16-byte halves
// of a 32-byte k-step). No barrier, no tile geometry: the pixels of all images form one list. LDS holds what a wave keeps to
// itself, its channels' parameters and its results on their way to whole rows. The four waves of
// a group are neighbours in (pixel tile, channel group) order with the channel group running fastest, so the waves that
// read the same pixels sit on one CU; the pixel rows come from HBM once and from the caches after that.
//
// Arithmetic and roundings are the general kernel's (conv_igemm.hip, general epilogue): float32 accumulation in
// v_mfma_f32_32x32x16_f16, bias, activation, the optional shortcut added to the value rounded to half, ReLU / the
// activation layer behind the convolution applied to the rounded half, one final rounding. (The split form adds its waves' sums
// in an order of its own, the same every time.)
//
// The int8 layer (DT == EXHIP_I8) is the same kernel on the same byte geometry -- a 32-byte k-step is 32 int8 channels,
// v_mfma_i32_32x32x32_i8 on the same 16-byte fragments -- with the int8 epilogue of the general kernel: dequantization
// fmaf((float)acc, scale, bias), activation, float32 shortcut, ReLU / activation layer, float32 NHWC and / or
// requantized int8 NHWC results.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "conv_pw_epilogue.h"
#include "conv_staged.h"
#include "pair.h"

namespace {

// U: k-steps per request round; two rounds are in flight. PAIRS: the pixels in 64-byte pieces, as in the split form below.
constexpr int pw_wave_lds(int dt, int mt, int nt, bool pairs) { return param_bytes(mt) + (pairs && nt * 4096 > tile_bytes(dt, mt) ? nt * 4096 : tile_bytes(dt, mt)); }
// (the kernel's group `bid` of `groups`)
template <int DT, int MT, int NT, int U, bool TAPS, bool PAIRS, typename EP>
__device__ __forceinline__ void pw_group(const PwParams& p, char* lds_all, unsigned bid, unsigned groups) {
    constexpr int OWN = pw_wave_lds(DT, MT, NT, PAIRS);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // workgroup ids are dealt round-robin to the 8 XCDs: give each XCD one contiguous run of items, so that the channel
    // groups of a pixel tile (and the weights' re-reads) share that XCD's L2
    {
        const unsigned per = groups >> 3;
        if (bid < (per << 3)) bid = (bid & 7) * per + (bid >> 3);
    }
    const unsigned item = __builtin_amdgcn_readfirstlane(bid * 4 + wave);
    if (item >= p.items) return;  // wave-uniform; the kernel has no barrier
    const unsigned tile = __builtin_amdgcn_readfirstlane(exhip_divide(item, p.ch_groups, p.groups_magic, p.groups_shift));
    const int kb0 = __builtin_amdgcn_readfirstlane((int)(item - tile * p.ch_groups) * MT);  // first 32-channel block
    char* const lds = lds_all + wave * OWN;

    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(p.x), 0, (int)p.x_bytes, kRsrcWord3);
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(p.wp), 0, (int)p.w_bytes, kRsrcWord3);

    // What a lane requests of the pixels. PAIRS: two k-steps at a time, 64 bytes of every pixel; four lanes read a pixel's, sixteen
    // pixels a load. Else a k-step at a time: the lane's pixel is lane & 31, its 16-byte half lane >> 5.
    constexpr int XL = PAIRS ? 2 : 1;
    int xoff[NT][XL];
    unsigned taps_in[NT][XL];  // TAPS: bit r * kw + q set where that tap of the pixel lies inside the image
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int l = 0; l < XL; ++l) {
            const unsigned pix = (tile * NT + nt) * 32 + (PAIRS ? l * 16 + (lane >> 2) : lane & 31);
            const int byte = (PAIRS ? lane & 3 : lane >> 5) * 16;
            if constexpr (TAPS) {
                // the filter's top-left input pixel; its offset may lie in front of the tensor (padding), the taps inside the
                // image never do, and 32-bit wrap-around of the sum gives their offsets
                const unsigned per_image = (unsigned)(p.out_h * p.out_w);
                const unsigned place = EP::pool ? pix >> 2 : pix;
                const unsigned img = exhip_divide(place, per_image, p.image_magic, p.image_shift), rem = place - img * per_image;
                int oy = (int)exhip_divide(rem, (unsigned)p.out_w, p.width_magic, p.width_shift), ox = (int)(rem - (unsigned)oy * (unsigned)p.out_w);
                if constexpr (EP::pool) {
                    oy = 2 * oy + (int)(pix >> 1 & 1);
                    ox = 2 * ox + (int)(pix & 1);
                }
                const int iy = oy * p.stride - p.pad_t, ix = ox * p.stride - p.pad_l;
                xoff[nt][l] = (((int)img * p.in_h + iy) * p.in_w + ix) * p.xs_b + byte;
                unsigned row = 0, m = 0;
                for (int q = 0; q < p.kw; ++q)
                    if ((unsigned)(ix + q) < (unsigned)p.in_w) row |= 1u << q;
                for (int r = 0; r < p.kh; ++r)
                    if ((unsigned)(iy + r) < (unsigned)p.in_h) m |= row << (r * p.kw);
                taps_in[nt][l] = pix < p.pixels ? m : 0;
            } else {
                xoff[nt][l] = pix < p.pixels ? (int)(pix * (unsigned)p.xs_b) + byte : kOutOfRange;
            }
        }
    // weight fragments: block kb of slab kb / mts lies at ((slab * n_ksteps + ks) * mts + kb % mts) KiB; the MT blocks
    // of a wave are neighbours in one slab (mts, 2 or 4, is a multiple of MT)
    const int w_step = p.mts * 1024, slab = kb0 >> (p.mts >> 1);
    const int w_base = (slab * p.n_ksteps * p.mts + (kb0 & (p.mts - 1))) * 1024;
    const int woff = lane * 16;

    typedef typename std::conditional<DT == EXHIP_I8, v16i, v16f>::type acc_t;
    acc_t acc[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[m][n][e] = 0;

    v4i a[2][U][MT], b[2][U][NT];
    const int nks = p.n_ksteps;
    // The request behind an odd last k-step reads the next row or block (or zeros beyond the view) and is not used.
    auto request = [&](auto buf_c, int ks0) {
        constexpr int buf = decltype(buf_c)::value;
#pragma unroll
        for (int u = 0; u < U; u += XL) {
            if (ks0 + (u & ~1) >= nks) continue;
            const int at = (ks0 + u) / XL < kMaxDirectSteps ? (ks0 + u) / XL : 0, entry = TAPS ? p.step[at] : 0;
            const int ws = TAPS && PAIRS ? p.pair_first[at] : ks0 + u;
#pragma unroll
            for (int l = 0; l < XL; ++l)
#pragma unroll
                for (int m = 0; m < MT; ++m)
                    a[buf][u + l][m] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(wr, woff + m * 1024, w_base + (ws + l * (PAIRS ? p.pair_w : 0)) * w_step, 0));
            const int off = entry & ((1 << kTapShift) - 1);
            const unsigned bit = 1u << ((unsigned)entry >> kTapShift);
#pragma unroll
            for (int l = 0; l < XL; ++l)
#pragma unroll
                for (int n = 0; n < NT; ++n) {
                    if constexpr (TAPS)
                        b[buf][u + l][n] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(xr, (taps_in[n][l] & bit) ? xoff[n][l] + off : kOutOfRange, 0, 0));
                    else
                        b[buf][u + l][n] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(xr, xoff[n][l], (ks0 + u) * 32, 0));
                }
        }
    };
    auto step = [&](auto buf_c, int u, const v4i (&xb)[NT]) {
        constexpr int buf = decltype(buf_c)::value;
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int n = 0; n < NT; ++n) {
                if constexpr (DT == EXHIP_I8)
                    acc[m][n] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[buf][u][m], xb[n], acc[m][n], 0, 0, 0);
                else
                    acc[m][n] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, a[buf][u][m]), __builtin_bit_cast(v8h, xb[n]),
                                                                       acc[m][n], 0, 0, 0);
            }
    };
    // PAIRS: four k-steps at a time through the wave's own LDS, from four lanes a pixel to one
    char* const stage_in = lds + param_bytes(MT) + (lane >> 2) * 64 + ((lane & 3) ^ (lane >> 3 & 3)) * 16;
    const char* const stage_out = lds + param_bytes(MT) + (lane & 31) * 64;
    // one round's products, of its k-steps below `left`
    auto products = [&](auto buf_c, int left) {
        constexpr int buf = decltype(buf_c)::value;
        if constexpr (PAIRS) {
#pragma unroll
            for (int u0 = 0; u0 < U; u0 += 4) {
                if (u0 >= left) continue;
                v4i x[4][NT];
#pragma unroll
                for (int u = 0; u < 4; ++u)
#pragma unroll
                    for (int n = 0; n < NT; ++n) *reinterpret_cast<v4i*>(stage_in + ((u >> 1) * NT + n) * 2048 + (u & 1) * 1024) = b[buf][u0 + u][n];
#pragma unroll
                for (int u = 0; u < 4; ++u)
#pragma unroll
                    for (int n = 0; n < NT; ++n)
                        x[u][n] = *reinterpret_cast<const v4i*>(stage_out + ((u >> 1) * NT + n) * 2048 + (((2 * (u & 1) + (lane >> 5)) ^ (lane >> 1 & 3)) * 16));
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (u < 2 || u0 + 2 < left) step(buf_c, u0 + u, x[u]);
            }
        } else {
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (u < left) step(buf_c, u, b[buf][u]);
        }
    };
    using B0 = std::integral_constant<int, 0>;
    using B1 = std::integral_constant<int, 1>;
    request(B0{}, 0);
    // the channels' parameters: lane = channel of the wave's MT * 32, zeros beyond K and for an absent array
    float par[kParams] = {};
    {
        const int at = (kb0 * 32 + lane) * 4;
        auto load = [&](const float* src, int offset, int count) {
            const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(src), 0, src ? count * 4 : 0, kRsrcWord3);
            return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, offset, 0, 0));
        };
        if constexpr (DT == EXHIP_I8) par[0] = load(p.scale, at, p.K);
        par[1] = load(p.bias, at, p.K);
        if (EP::any || EP::post == kPostPrelu) par[2] = load(p.post_slope, p.post_slope_shared ? 0 : at, p.post_slope_shared ? 1 : p.K);
        if (DT == EXHIP_I8 && (EP::any ? p.post_bn_a != nullptr : EP::bn)) {
            par[2] = load(p.post_bn_a, at, p.K);
            par[3] = load(p.post_bn_b, at, p.K);
        }
    }
    request(B1{}, U);
    int ks0 = 0;
    for (; ks0 + 2 * U < nks; ks0 += 2 * U) {
        products(B0{}, U);
        request(B0{}, ks0 + 2 * U);
        products(B1{}, U);
        request(B1{}, ks0 + 3 * U);
    }
    // (the loop leaves with both rounds of the last 2 * U k-steps requested)
    if (MT == 2 || lane < 32) {
#pragma unroll
        for (int i = 0; i < kParams; ++i) *reinterpret_cast<float*>(lds + (i * MT * 32 + lane) * 4) = par[i];
    }
    products(B0{}, nks - ks0);
    products(B1{}, nks - ks0 - U);
    pw_epilogue<DT, MT, NT, EP>(p, acc, tile * NT * 32, p.pixels, kb0, lane, lds);
}

template <int DT, int MT, int NT, int U, bool TAPS, bool PAIRS, typename EP>
__global__ __launch_bounds__(256, 2) void conv1x1_pw_kernel(const PwParams p) {
    exhip_touch_args(p);
    __shared__ __attribute__((aligned(16))) char lds_all[4 * pw_wave_lds(DT, MT, NT, PAIRS)];
    pw_group<DT, MT, NT, U, TAPS, PAIRS, EP>(p, lds_all, blockIdx.x, gridDim.x);
}

// The split form, for launches of few tiles and many k-steps (one image, deep layers), where the kernel above is as long as one
// wave's chain: 0.17 us a k-step, 16 us for 256 -> 256 3x3 int8 on a 20 x 20 map. WK waves share a tile of 32 pixels x 32 * MT
// channels: each takes its run of the k-steps, the sums meet in LDS (exactly for int8; in a fixed order, so the same bits
// every time, for fp16), and each wave finishes its quarter of the tile, eight channels of a pixel per lane (wave m the whole block m
// where the layers behind are looked at at run time: a head's groups take 32 channels at a time). Every request in the loop is unconditional, so that the waits count what is in
// flight; those past a wave's run ask for operands it does not use.
template <int DT, int MT, int WK, typename EP>
constexpr int split_lds() { return WK * MT * 4096 + (EP::any ? MT * wave_bytes(DT, 1) : WK * param_bytes(1)); }
template <int DT, int MT, int WK, bool TAPS, bool PAIRS, typename EP>
__device__ __forceinline__ void split_group(const PwParams& p, char* lds_all, unsigned item, unsigned groups) {
    constexpr int R = 8;  // k-steps in flight
    constexpr bool I8 = DT == EXHIP_I8;
    constexpr int RED = WK * MT * 4096;
    constexpr int OWN = EP::any ? wave_bytes(DT, 1) : param_bytes(1);
    static_assert(MT == 2 && WK == 4 && WK <= kSplit, "two waves finish a block");
    const int lane = threadIdx.x & 63, part = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    {
        const unsigned per = groups >> 3;
        if (item < (per << 3)) item = (item & 7) * per + (item >> 3);
    }
    const unsigned tile = __builtin_amdgcn_readfirstlane(exhip_divide(item, p.ch_groups, p.groups_magic, p.groups_shift));
    const int kb0 = __builtin_amdgcn_readfirstlane((int)(item - tile * p.ch_groups) * MT);
    const int own_block = EP::any ? part : part >> 1;   // the block the wave finishes, or half of it
    const bool finishes = own_block < MT;
    char* const lds = lds_all + RED + (finishes ? part : 0) * OWN;
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(p.x), 0, (int)p.x_bytes, kRsrcWord3);
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(p.wp), 0, (int)p.w_bytes, kRsrcWord3);

    // What a lane requests of the pixels. PAIRS: two k-steps at a time, 64 bytes of every pixel; four lanes read a pixel's, sixteen
    // pixels a load. Else a k-step at a time: the lane's pixel is lane & 31, its 16-byte half lane >> 5.
    constexpr int XL = PAIRS ? 2 : 1;
    int xoff[XL], iy[XL], ix[XL];
#pragma unroll
    for (int j = 0; j < XL; ++j) {
        const unsigned pix = tile * 32 + (PAIRS ? j * 16 + (lane >> 2) : lane & 31);
        const int byte = (PAIRS ? lane & 3 : lane >> 5) * 16;
        if constexpr (TAPS) {
            const unsigned per_image = (unsigned)(p.out_h * p.out_w);
            const unsigned img = exhip_divide(pix, per_image, p.image_magic, p.image_shift), rem = pix - img * per_image;
            const int oy = (int)exhip_divide(rem, (unsigned)p.out_w, p.width_magic, p.width_shift), ox = (int)(rem - (unsigned)oy * (unsigned)p.out_w);
            iy[j] = oy * p.stride - p.pad_t;
            ix[j] = ox * p.stride - p.pad_l;
            xoff[j] = (((int)img * p.in_h + iy[j]) * p.in_w + ix[j]) * p.xs_b + byte;
            if (pix >= p.pixels) iy[j] = -0x40000000;
        } else {
            xoff[j] = pix < p.pixels ? (int)(pix * (unsigned)p.xs_b) + byte : kOutOfRange;
        }
    }
    const int s_first = PAIRS ? p.start_w[part] : p.start_s[part], steps = p.start_s[part + 1] - p.start_s[part];
    const int pair_w = PAIRS ? p.pair_w : 0, s_last = p.n_ksteps - 1 - pair_w;
    const int w_step = p.mts * 1024, slab = kb0 >> (p.mts >> 1);
    const int w_base = (slab * p.n_ksteps * p.mts + (kb0 & (p.mts - 1))) * 1024;
    int s_at = s_first, b_at = p.start_b[part], r_at = p.start_r[part], q_at = p.start_q[part], left = p.start_left[part];
    int xcur[XL];
    auto enter_tap = [&]() {  // the lane's offsets at the tap, out of range outside the image
#pragma unroll
        for (int j = 0; j < XL; ++j) {
            const bool in = (unsigned)(iy[j] + r_at) < (unsigned)p.in_h && (unsigned)(ix[j] + q_at) < (unsigned)p.in_w;
            xcur[j] = in ? xoff[j] + b_at : kOutOfRange;
        }
    };
#pragma unroll
    for (int j = 0; j < XL; ++j) xcur[j] = xoff[j];
    if constexpr (TAPS) enter_tap();

    typedef typename std::conditional<DT == EXHIP_I8, v16i, v16f>::type acc_t;
    acc_t acc[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[m][e] = 0;
    v4i a[R][MT], b[R];
    auto request = [&](int u) {  // PAIRS: k-steps u and u + 1, u even
        const int s_in = s_at < s_last ? s_at : s_last;
#pragma unroll
        for (int j = 0; j < XL; ++j) {
            b[u + j] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(xr, xcur[j], TAPS ? 0 : s_in * 32, 0));
#pragma unroll
            for (int m = 0; m < MT; ++m)
                a[u + j][m] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(wr, lane * 16 + m * 1024, w_base + (s_in + j * pair_w) * w_step, 0));
        }
        s_at += PAIRS ? p.next_w : 1;
        if constexpr (TAPS) {
            b_at += 32 * XL;
            left -= 32 * XL;
            if (left == 0) {  // the next tap (no memory accesses under the branch)
                left = p.chunk_b;
                b_at += p.xs_b - p.chunk_b;
                if (++q_at == p.kw) {
                    q_at = 0;
                    b_at += p.row_end_b;
                    if (++r_at == p.kh) {
                        r_at = 0;
                        b_at += p.chunk_end_b;
                        if (PAIRS) s_at += p.chunk_w;
                    }
                }
                enter_tap();
            } else {
#pragma unroll
                for (int j = 0; j < XL; ++j) xcur[j] += xcur[j] == kOutOfRange ? 0 : 32 * XL;
            }
        }
    };
    // PAIRS: through the wave's own LDS from four lanes a pixel to one. A CU takes 16 cycles for a load whose neighbouring lanes read
    // 64 bytes of a pixel, up to 64 for one whose lanes read pixels a power of two apart, and a short launch spends its time on
    // the requests (256 -> 256 3x3 int8 on one 20 x 20 map: 3400 cycles of 12 500 until the last of the first eight k-steps' is out).
    // A pixel's 16-byte columns are dealt out by its number, so that neither side meets bank conflicts.
    char* const stage = lds_all + part * MT * 4096;
    char* const stage_in = stage + (lane >> 2) * 64 + ((lane & 3) ^ (lane >> 3 & 3)) * 16;   // (pixel >> 1) & 3, for either load
    const char* const stage_out = stage + (lane & 31) * 64;
    v4i x[2][2];
    auto arrange = [&](int u, int to) {
#pragma unroll
        for (int j = 0; j < 2; ++j) *reinterpret_cast<v4i*>(stage_in + j * 1024) = b[u + j];
#pragma unroll
        for (int j = 0; j < 2; ++j) x[to][j] = *reinterpret_cast<const v4i*>(stage_out + (((2 * j + (lane >> 5)) ^ (lane >> 1 & 3)) * 16));
    };
    auto product = [&](int u, const v4i& xb) {
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            if constexpr (DT == EXHIP_I8) acc[m] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[u][m], xb, acc[m], 0, 0, 0);
            else acc[m] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, a[u][m]), __builtin_bit_cast(v8h, xb), acc[m], 0, 0, 0);
        }
    };
    float par[kParams] = {};
    auto load_parameters = [&]() {  // of the block this wave will finish: lane = channel
        const int at = lane < 32 ? ((kb0 + own_block) * 32 + lane) * 4 : kOutOfRange;
        auto load = [&](const float* src, int offset, int count) {
            const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(src), 0, src ? count * 4 : 0, kRsrcWord3);
            return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, offset, 0, 0));
        };
        if constexpr (DT == EXHIP_I8) par[0] = load(p.scale, at, p.K);
        par[1] = load(p.bias, at, p.K);
        if (EP::any || EP::post == kPostPrelu) par[2] = load(p.post_slope, p.post_slope_shared ? 0 : at, p.post_slope_shared ? 1 : p.K);
        if (DT == EXHIP_I8 && (EP::any ? p.post_bn_a != nullptr : EP::bn)) {
            par[2] = load(p.post_bn_a, at, p.K);
            par[3] = load(p.post_bn_b, at, p.K);
        }
    };
    auto step = [&](int u) {  // k-step u; PAIRS: the pair, whose pixels have been arranged
        if constexpr (PAIRS) {
            product(u, x[u / 2 & 1][0]);
            product(u + 1, x[u / 2 & 1][1]);
        } else {
            product(u, b[u]);
        }
    };
    if (steps > R) {
#pragma unroll
        for (int u = 0; u < R; u += XL) request(u);
        if constexpr (PAIRS) arrange(0, 0);
        int k = 0;
        for (; k + R < steps; k += R) {
#pragma unroll
            for (int u = 0; u < R; u += XL) {
                if constexpr (PAIRS) arrange((u + 2) % R, (u / 2 + 1) & 1);
                step(u);
                request(u);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (finishes) load_parameters();
#pragma unroll
        for (int u = 0; u < R; u += XL)
            if (k + u < steps) {
                if constexpr (PAIRS)
                    if (u + 2 < R) arrange(u + 2, (u / 2 + 1) & 1);
                step(u);
            }
    } else {
#pragma unroll
        for (int u = 0; u < R; u += XL)
            if (u < steps) request(u);
        if (finishes) load_parameters();
#pragma unroll
        for (int u = 0; u < R; u += XL)
            if (u < steps) {
                if constexpr (PAIRS) arrange(u, u / 2 & 1);
                step(u);
            }
    }
    // the waves' sums: 16 words a lane and block, 16 bytes side by side per lane
    auto word4 = [](const acc_t& c, int q) {
        if constexpr (DT == EXHIP_I8) return v4i{c[q * 4], c[q * 4 + 1], c[q * 4 + 2], c[q * 4 + 3]};
        else return __builtin_bit_cast(v4i, v4f{c[q * 4], c[q * 4 + 1], c[q * 4 + 2], c[q * 4 + 3]});
    };
    const int k_end = pw_channel_end(p.K, p.kstride, p.exact), half = lane >> 5, row = lane & 31, kb = kb0 + own_block;
    const int rows = p.pixels - tile * 32 < 32 ? (int)(p.pixels - tile * 32) : 32;
    constexpr int N = 8, RV = I8 ? 2 : 1;   // channels a lane, 16-byte pieces of their shortcut
    const int ch = half * 16 + (part & 1) * N;   // of the block's
    v4i res[RV];
    if constexpr (!EP::any && EP::res != 0) {
        const int row_b = p.kstride * (I8 ? 4 : 2), ch_b = I8 ? 4 : 2;
        const __amdgpu_buffer_rsrc_t rr = tile_view(I8 ? (const void*)p.residual_f : (const void*)p.residual, tile * 32, row_b, kb * 32 * ch_b, rows);
#pragma unroll
        for (int q = 0; q < RV; ++q)
            res[q] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rr, pw_lane_offset(row, row_b, ch * ch_b + q * 16, (p.kstride - kb * 32) * ch_b), 0, 0));
    }
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int q = 0; q < 4; ++q) *reinterpret_cast<v4i*>(lds_all + (part * MT + m) * 4096 + q * 1024 + lane * 16) = word4(acc[m], q);
    __syncthreads();
    // what finishes a second block that does not exist (an odd number of blocks) is done too
    if (!finishes || !pw_block_exists(kb, k_end)) return;
    if (lane < 32) {
#pragma unroll
        for (int i = 0; i < kParams; ++i) *reinterpret_cast<float*>(lds + (i * 32 + lane) * 4) = par[i];
    }
    auto sum4 = [&](int q, auto* to) {  // four channels' sums over the waves
        v4i t = *reinterpret_cast<const v4i*>(lds_all + own_block * 4096 + q * 1024 + lane * 16);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if constexpr (I8) to[e] = t[e];
            else to[e] = __builtin_bit_cast(v4f, t)[e];
        }
#pragma unroll
        for (int w = 1; w < WK; ++w) {
            t = *reinterpret_cast<const v4i*>(lds_all + (w * MT + own_block) * 4096 + q * 1024 + lane * 16);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if constexpr (I8) to[e] += t[e];
                else to[e] += __builtin_bit_cast(v4f, t)[e];
            }
        }
    };
    typename std::conditional<I8, int, float>::type total[EP::any ? 16 : N];
#pragma unroll
    for (int q = 0; q < (EP::any ? 4 : N / 4); ++q) sum4(EP::any ? q : (part & 1) * (N / 4) + q, total + q * 4);
    if constexpr (EP::any) {
        acc_t sum[1][1];
#pragma unroll
        for (int e = 0; e < 16; ++e) sum[0][0][e] = total[e];
        pw_epilogue<DT, 1, 1, EP>(p, sum, tile * 32, p.pixels, kb, lane, lds);
    } else {
        float v[N], scale[N], bias[N];
        if constexpr (I8) read_parameters<1>(lds, 0, ch, scale);
        read_parameters<1>(lds, 1, ch, bias);
#pragma unroll
        for (int e = 0; e < N; ++e) {
            if constexpr (I8) v[e] = __builtin_fmaf((float)total[e], scale[e], bias[e]);
            else v[e] = total[e] + bias[e];
        }
        layers_behind<DT, 1, EP>(p, v, lds, ch, EP::res != 0, [&](int e) {
            const int word = res[I8 ? e >> 2 : 0][I8 ? e & 3 : e >> 1];
            if constexpr (I8) return __builtin_bit_cast(float, word);
            else return exhip_h2f((uint16_t)(((uint32_t)word >> ((e & 1) * 16)) & 0xffff));
        });
        if (kb * 32 + 32 > p.K) {  // pad channels hold zeros
#pragma unroll
            for (int e = 0; e < N; ++e)
                if (kb * 32 + ch + e >= p.K) v[e] = 0.f;
        }
        typedef unsigned v4u __attribute__((ext_vector_type(4)));
        typedef unsigned v2u __attribute__((ext_vector_type(2)));
        if constexpr (I8) {
            if (p.y_f) {
                const __amdgpu_buffer_rsrc_t y = tile_view(p.y_f, tile * 32, p.kstride * 4, kb * 128, rows);
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    const v4f o = {v[q * 4], v[q * 4 + 1], v[q * 4 + 2], v[q * 4 + 3]};
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, o), y, pw_lane_offset(row, p.kstride * 4, ch * 4 + q * 16, (k_end - kb * 32) * 4), 0, 0);
                }
            }
            if (p.y_q) {
                v2u o;
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    uint32_t w = 0;
#pragma unroll
                    for (int e = 0; e < 4; ++e) w |= (uint32_t)(exhip_q8(v[q * 4 + e] * p.fs_out) & 0xff) << (8 * e);
                    o[q] = w;
                }
                __builtin_amdgcn_raw_buffer_store_b64(o, tile_view(p.y_q, tile * 32, p.kstride, kb * 32, rows), pw_lane_offset(row, p.kstride, ch, k_end - kb * 32), 0, 0);
            }
        } else {
            const v4u o = {exhip_round_pair(v[0], v[1]), exhip_round_pair(v[2], v[3]), exhip_round_pair(v[4], v[5]), exhip_round_pair(v[6], v[7])};
            __builtin_amdgcn_raw_buffer_store_b128(o, tile_view(p.y, tile * 32, p.kstride * 2, kb * 64, rows), pw_lane_offset(row, p.kstride * 2, ch * 2, (k_end - kb * 32) * 2), 0, 0);
        }
    }
}

template <int DT, int MT, int WK, bool TAPS, bool PAIRS, typename EP>
__global__ __launch_bounds__(64 * WK, 2) void conv_pw_split_kernel(const PwParams p) {
    exhip_touch_args(p);
    __shared__ __attribute__((aligned(16))) char lds_all[split_lds<DT, MT, WK, EP>()];
    split_group<DT, MT, WK, TAPS, PAIRS, EP>(p, lds_all, blockIdx.x, gridDim.x);
}

// Two pointwise layers that do not read each other's results in one launch, each in its own form: a bottleneck's last layer and the one beside it, on the
// two inputs of a Concat. Launched one after the other each waits for the other's last group, and at one image each is 4 us whatever it computes:
// 64 -> 64 and 128 -> 64 at 1 x 80 x 80 int8 7.7 us, here 4.2, at 16 x 80 x 80 15.0 and 12.1; fp16 7.1 and 3.5, 16.2 and 13.2. No pair of eight sizes took longer.
struct PwTwo {
    PwParams p[2];
    int kind[2];
    unsigned groups[2];
};
constexpr int kTwoLds = 34816;
template <int DT>  // what stands behind them in the networks: int8 a BatchNorm and a LeakyReLU layer (through the Concat), fp16 nothing
using TwoEp = typename std::conditional<DT == EXHIP_I8, Ep<0, kPostLeaky, 0, true>, Ep<0, kPostNone, 0>>::type;
// the forms by number, -1 for all others
template <int DT, int MT, int NT, int U, bool TAPS, typename EP>
constexpr int two_kind() {
    if (TAPS || !std::is_same<EP, TwoEp<DT>>::value) return -1;
    if (MT == 1 && NT == 2) return U == 4 ? 0 : U == 104 ? 1 : -1;
    return MT != 2 || NT != 1 ? -1 : U == 4 ? 2 : U == 104 ? 3 : U == -2 * kSplit ? 4 : -1;
}
template <int DT>
__device__ __forceinline__ void two_group(const PwParams& p, int kind, char* lds, unsigned bid, unsigned groups) {
    exhip_touch_args(p);
    if (kind == 0) pw_group<DT, 1, 2, 4, false, false, TwoEp<DT>>(p, lds, bid, groups);
    else if (kind == 1) pw_group<DT, 1, 2, 4, false, true, TwoEp<DT>>(p, lds, bid, groups);
    else if (kind == 2) pw_group<DT, 2, 1, 4, false, false, TwoEp<DT>>(p, lds, bid, groups);
    else if (kind == 3) pw_group<DT, 2, 1, 4, false, true, TwoEp<DT>>(p, lds, bid, groups);
    else split_group<DT, 2, kSplit, false, true, TwoEp<DT>>(p, lds, bid, groups);
}
template <int DT>
__global__ __launch_bounds__(256, 2) void conv_pw_two_kernel(const PwTwo q) {
    static_assert(4 * pw_wave_lds(DT, 1, 2, true) <= kTwoLds && 4 * pw_wave_lds(DT, 2, 1, true) <= kTwoLds && split_lds<DT, 2, kSplit, TwoEp<DT>>() <= kTwoLds, "one LDS for all");
    __shared__ __attribute__((aligned(16))) char lds[kTwoLds];
    const unsigned first = q.groups[0];
    if (blockIdx.x < first) two_group<DT>(q.p[0], q.kind[0], lds, blockIdx.x, first);
    else two_group<DT>(q.p[1], q.kind[1], lds, blockIdx.x - first, q.groups[1]);
}

// A depthwise 3x3 layer and the pointwise layer that alone reads it, the depthwise results staying in LDS. A group computes
// all C channels of dw_pixels output pixels -- a thread owns four channels of strips of PX pixels, the arithmetic and roundings
// of dwconv3x3_nhwc_strip_kernel -- and its four waves then take the pixels' 32 x 32 output blocks (of fewer than 32 pixels the
// block's other columns repeat them and are not stored), pixel fragments from LDS, weight fragments from L2 with R k-steps in flight;
// SMALL, a launch of few groups, asks for the first of them before the depthwise half. A small launch deals the output channels over
// several groups, each with depthwise results of its own. A layer that the split form above would take (dw_split) adds its four
// runs of k-steps in that form's order. Bound by the chain of one group where it is small (1 x 64 x 56 x 56 takes 3.9 us, 7.7 as two launches;
// 256 -> 128 at 1 x 14 x 14 5.2 and 8.2), by the depthwise loads where it is large (64 x 128 x 56 x 56 -> 64: 33.8 us and 47.5; 40.3 when
// every thread read its 36 weights by itself and 64 pixels a group were the most).
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef int v2i __attribute__((ext_vector_type(2)));

template <int S, int PX, bool SMALL, typename EP>
__global__ __launch_bounds__(256, 3) void dw_pw_kernel(const PwParams p) {
    exhip_touch_args(p);
    constexpr int R = 4, NC = (PX - 1) * S + 3;
    constexpr unsigned kRowOutside = 0x80000000u, kColOutside = 0x40000000u;  // tensors of at most 2^30 bytes: beyond the view, alone or together
    extern __shared__ __attribute__((aligned(16))) char lds_dyn[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    unsigned item0 = blockIdx.x;
    {
        const unsigned per = gridDim.x >> 3;
        if (item0 < (per << 3)) item0 = (item0 & 7) * per + (item0 >> 3);
    }
    const unsigned tile = __builtin_amdgcn_readfirstlane(exhip_divide(item0, p.ch_groups, p.groups_magic, p.groups_shift));
    const int kb_first = __builtin_amdgcn_readfirstlane((int)(item0 - tile * p.ch_groups) * p.dw_kblocks);
    const unsigned pix0 = tile * p.dw_pixels, pix_end = min(p.pixels, pix0 + p.dw_pixels);
    char* const lds = lds_dyn + wave * wave_bytes(EXHIP_F16, 1);
    char* const mid = lds_dyn + p.dw_mid;
    const int mid_pitch = p.xs_b + 16;
    const int nks = p.n_ksteps, w_step = p.mts * 1024;
    const int blocks = p.kblocks - kb_first < p.dw_kblocks ? p.kblocks - kb_first : p.dw_kblocks;
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(p.wp), 0, (int)p.w_bytes, kRsrcWord3);
    v4i a[R];
    float par[kParams] = {};
    auto weights_at = [&](int kb) { return ((kb >> (p.mts >> 1)) * nks * p.mts + (kb & (p.mts - 1))) * 1024; };
    auto request = [&](int w_base, int u, int s) {
        a[u] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(wr, lane * 16, w_base + (s < nks ? s : nks - 1) * w_step, 0));
    };
    auto load_parameters = [&](int kb) {
        const int at = lane < 32 ? (kb * 32 + lane) * 4 : kOutOfRange;
        auto load = [&](const float* src, int offset, int count) {
            const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(src), 0, src ? count * 4 : 0, kRsrcWord3);
            return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, offset, 0, 0));
        };
        par[1] = load(p.bias, at, p.K);
        if (EP::any || EP::post == kPostPrelu) par[2] = load(p.post_slope, p.post_slope_shared ? 0 : at, p.post_slope_shared ? 1 : p.K);
    };
    {
        const int groups = p.xs_b >> 3, g = threadIdx.x % groups, lanes = 256 / groups, first = threadIdx.x / groups;
        const int strips = first < lanes ? p.dw_pixels / PX : 0;
        const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(p.x), 0, (int)p.x_bytes, kRsrcWord3);
        const unsigned per_image = (unsigned)(p.out_h * p.out_w);
        const int row_b = p.in_w * p.xs_b;
        // The 36 weights of a thread's four channels lie 144 bytes from the next thread's: read so, each load is 64 lines and takes
        // its CU 64 cycles. The group's threads read them side by side instead and take their own from LDS.
        v4f* const wk = reinterpret_cast<v4f*>(lds_dyn);
        constexpr int kAhead = 2;   // 16-byte pieces a thread has in flight
        const int pieces = groups * 9;
        v4f piece[kAhead];
#pragma unroll
        for (int q = 0; q < kAhead; ++q) piece[q] = reinterpret_cast<const v4f*>(p.dw_w)[min((int)threadIdx.x + q * 256, pieces - 1)];
        float b[4] = {0.f, 0.f, 0.f, 0.f}, sl[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (p.dw_bias) b[e] = p.dw_bias[g * 4 + e];
            if (p.dw_slope) sl[e] = p.dw_slope[p.dw_slope_shared ? 0 : g * 4 + e];
        }
        auto load = [&](int st, v4h (&r)[3][NC]) {
            const unsigned pix = pix0 + st * PX;
            const unsigned img = exhip_divide(pix, per_image, p.image_magic, p.image_shift), rem = pix - img * per_image;
            const int oy = (int)exhip_divide(rem, (unsigned)p.out_w, p.width_magic, p.width_shift), ox = (int)(rem - (unsigned)oy * (unsigned)p.out_w);
            const int iy = pix < p.pixels && st < strips ? oy * S - p.pad_t : -4, ix = ox * S - p.pad_l;
            const unsigned at = img * (unsigned)(p.in_h * row_b) + g * 8;
            unsigned row_off[3], col_off[NC];
#pragma unroll
            for (int a = 0; a < 3; ++a) row_off[a] = (unsigned)(iy + a) < (unsigned)p.in_h ? at + (unsigned)((iy + a) * row_b) : kRowOutside;
#pragma unroll
            for (int c = 0; c < NC; ++c) col_off[c] = (unsigned)(ix + c) < (unsigned)p.in_w ? (unsigned)((ix + c) * p.xs_b) : kColOutside;
#pragma unroll
            for (int a = 0; a < 3; ++a)
#pragma unroll
                for (int c = 0; c < NC; ++c) r[a][c] = __builtin_bit_cast(v4h, __builtin_amdgcn_raw_buffer_load_b64(xr, (int)(row_off[a] + col_off[c]), 0, 0));
        };
        v4h r[3][NC];
        load(first, r);
        if constexpr (SMALL) {  // the pointwise layer's first weights are on their way while the depthwise results are made
            if (wave < blocks) {
#pragma unroll
                for (int u = 0; u < R; ++u) request(weights_at(kb_first + wave), u, u);
                load_parameters(kb_first + wave);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < kAhead; ++q)
            if ((int)threadIdx.x + q * 256 < pieces) wk[threadIdx.x + q * 256] = piece[q];
        for (int i = threadIdx.x + kAhead * 256; i < pieces; i += 256) wk[i] = reinterpret_cast<const v4f*>(p.dw_w)[i];
        __syncthreads();
        float k[36];
#pragma unroll
        for (int q = 0; q < 9; ++q) {
            const v4f t = wk[g * 9 + q];
#pragma unroll
            for (int e = 0; e < 4; ++e) k[q * 4 + e] = t[e];
        }
        auto compute = [&](int st, const v4h (&r)[3][NC]) {
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
                        for (int a = 0; a < 3; ++a) s = __builtin_fmaf((float)r[a][px * S + j][e], k[e * 9 + a * 3 + j], s);
                        sum += s;
                    }
                    res[e] = sum;
                }
                if (p.dw_slope) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float h = exhip_h2f(exhip_f2h(res[e]));
                        res[e] = h >= 0.f ? h : sl[e] * h;
                    }
                } else if (p.dw_act != 0) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        res[e] = (0.f > res[e]) ? 0.f : res[e];
                        if (p.dw_act == 3) res[e] = res[e] <= 6.f ? res[e] : 0.f;
                    }
                }
                const v2i o = {(int)exhip_round_pair(res[0], res[1]), (int)exhip_round_pair(res[2], res[3])};
                *reinterpret_cast<v2i*>(mid + (st * PX + px) * mid_pitch + g * 8) = o;
            }
        };
        for (int st = first; st < strips; st += lanes) {
            compute(st, r);
            if (st + lanes < strips) load(st + lanes, r);
        }
    }
    __syncthreads();
    for (int item = wave; item < blocks * p.dw_tiles; item += 4) {
        const int sub = item & (p.dw_tiles - 1), kb = kb_first + (item >> __builtin_ctz(p.dw_tiles));
        const unsigned first = pix0 + sub * 32;
        if (first >= p.pixels) continue;  // wave-uniform; no barrier follows
        const int w_base = weights_at(kb);
        if (!SMALL || item != wave) {
#pragma unroll
            for (int u = 0; u < R; ++u) request(w_base, u, u);
            load_parameters(kb);
        }
        v16f acc, sum[1][1];
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[e] = sum[0][0][e] = 0.f;
        const char* src = mid + (sub * 32 + (lane & 31 & (p.dw_pixels - 1))) * mid_pitch + (lane >> 5) * 16;
        int run = 1, end = p.dw_split ? p.start_s[1] : nks;
        for (int s = 0; s < nks; s += R) {
#pragma unroll
            for (int u = 0; u < R; ++u) {
                if (s + u < nks) {
                    if (s + u == end) {
#pragma unroll
                        for (int e = 0; e < 16; ++e) sum[0][0][e] += acc[e], acc[e] = 0.f;
                        do end = p.start_s[++run]; while (end == s + u);
                    }
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, a[u]), *reinterpret_cast<const v8h*>(src + (s + u) * 32), acc, 0, 0, 0);
                }
                request(w_base, u, s + R + u);
            }
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) sum[0][0][e] += acc[e];
        if (lane < 32) {
#pragma unroll
            for (int i = 0; i < kParams; ++i) *reinterpret_cast<float*>(lds + (i * 32 + lane) * 4) = par[i];
        }
        pw_epilogue<EXHIP_F16, 1, 1, EP>(p, sum, first, pix_end, kb, lane, lds);
    }
}

// ---- the first layer of a network: 3x3 on the planes of at most four channels, with the Input layer in front ----
// Halves for an fp16 network, float32 for an int8 one, whose quantizer is in here as well. A group takes tile_rows whole output rows of an image, which are
// neighbouring pixels of the NHWC result. It reads the input rows they need from the planes (VEC: eight pixels at a time), applies (x - mean) * factor, rounds
// to half as the Input layer does or quantizes, and leaves pixels of four halves or bytes in LDS, padding as zeros; a filter row is then one
// k-step, a lane's 16 bytes two or four neighbouring taps. The weights are the general kernel's packed first-layer form, the order of the sums is its as well. Bound by the stores of the result in a large launch (3 -> 64 at stride 2
// with the Input layer, 64 x 224 x 224: 26 us, 103 MB; 81 as Input layer, conversion and convolution, 61 the convolution alone), by the
// launch in a small one (1 x 112 x 112: 4.0, 16.0 and 11.4); the int8 form 3 -> 16 at 64 x 128 x 128 takes 24.6 us, 70 as Input layer, quantizer (11.3) and convolution.
// Rows of a width that is no multiple of eight cost two-byte loads (64 x 223 x 223: 34 us, 142).
template <int DT, int MT, bool VEC, typename EP>
__global__ __launch_bounds__(256, EP::any ? 2 : 4) void stem_planes_kernel(const PwParams p) {
    exhip_touch_args(p);
    constexpr bool I8 = DT == EXHIP_I8;
    constexpr int KH = 3;
    typedef typename std::conditional<I8, int, v2i>::type pixel_t;
    typedef typename std::conditional<I8, float, uint16_t>::type plane_t;
    extern __shared__ __attribute__((aligned(16))) char lds_dyn[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    unsigned item0 = blockIdx.x;
    {
        const unsigned per = gridDim.x >> 3;
        if (item0 < (per << 3)) item0 = (item0 & 7) * per + (item0 >> 3);
    }
    const unsigned img = __builtin_amdgcn_readfirstlane(exhip_divide(item0, p.ch_groups, p.groups_magic, p.groups_shift));
    const int oy0 = __builtin_amdgcn_readfirstlane((int)(item0 - img * p.ch_groups) * p.tile_rows);
    const int rows = min(p.tile_rows, p.out_h - oy0), in_rows = (rows - 1) * p.stride + KH, iy0 = oy0 * p.stride - p.pad_t;
    char* const lds = lds_dyn + wave * wave_bytes(DT, MT);
    pixel_t* const px = reinterpret_cast<pixel_t*>(lds_dyn + 4 * wave_bytes(DT, MT));

    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(p.wp), 0, (int)p.w_bytes, kRsrcWord3);
    v4i a[KH][MT];
    float par[kParams] = {};
    auto load_block = [&](int kb) {
        const int w_base = ((kb >> (p.mts >> 1)) * KH * p.mts + (kb & (p.mts - 1))) * 1024;
#pragma unroll
        for (int r = 0; r < KH; ++r)
#pragma unroll
            for (int m = 0; m < MT; ++m)
                a[r][m] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(wr, lane * 16, w_base + (r * p.mts + m) * 1024, 0));
        const int at = MT == 2 || lane < 32 ? (kb * 32 + lane) * 4 : kOutOfRange;
        auto load = [&](const float* src, int offset, int count) {
            const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(src), 0, src ? count * 4 : 0, kRsrcWord3);
            return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, offset, 0, 0));
        };
        if constexpr (I8) par[0] = load(p.scale, at, p.K);
        par[1] = load(p.bias, at, p.K);
        if (EP::any || EP::post == kPostPrelu) par[2] = load(p.post_slope, p.post_slope_shared ? 0 : at, p.post_slope_shared ? 1 : p.K);
    };

    const int plane = p.in_h * p.in_w;
    const plane_t* const image = reinterpret_cast<const plane_t*>(p.x) + (size_t)img * p.in_c * plane;
    auto scaled = [&](float v, int c) { return p.mean ? (v - p.mean[c]) * p.factor[c] : v; };
    if constexpr (VEC) {
        typedef float v8f __attribute__((ext_vector_type(8)));
        for (int i = threadIdx.x; i < in_rows * p.pieces; i += 256) {
            const int r = (int)exhip_divide((unsigned)i, (unsigned)p.pieces, p.pieces_magic, p.pieces_shift), x8 = i - r * p.pieces, iy = iy0 + r;
            const bool inside = (unsigned)iy < (unsigned)p.in_h;
            pixel_t* const to = px + r * p.row_pixels + p.pad_l + x8 * 8;
            if constexpr (I8) {
                v4f v[4][2] = {};
                if (inside) {
#pragma unroll
                    for (int c = 0; c < 4; ++c)
                        if (c < p.in_c) {
                            const v4f* const from = reinterpret_cast<const v4f*>(image + (size_t)c * plane + iy * p.in_w + x8 * 8);
                            v[c][0] = from[0];
                            v[c][1] = from[1];
                        }
                }
                int word[8] = {};
                if (inside) {
#pragma unroll
                    for (int c = 0; c < 4; ++c)
                        if (c < p.in_c) {
#pragma unroll
                            for (int e = 0; e < 8; ++e) word[e] |= (int)((unsigned)(exhip_q8(scaled(v[c][e >> 2][e & 3], c) * p.fs_in) & 0xff) << (8 * c));
                        }
                }
#pragma unroll
                for (int e = 0; e < 8; ++e) to[e] = word[e];
            } else {
                v4i v[4] = {};
                if (inside) {
#pragma unroll
                    for (int c = 0; c < 4; ++c)
                        if (c < p.in_c) v[c] = *reinterpret_cast<const v4i*>(image + (size_t)c * plane + iy * p.in_w + x8 * 8);
                    if (p.mean) {
#pragma unroll
                        for (int c = 0; c < 4; ++c)
                            if (c < p.in_c) {
                                v8f f = __builtin_convertvector(__builtin_bit_cast(v8h, v[c]), v8f);
#pragma unroll
                                for (int e = 0; e < 8; ++e) f[e] = (f[e] - p.mean[c]) * p.factor[c];
                                v[c] = __builtin_bit_cast(v4i, __builtin_convertvector(f, v8h));
                            }
                    }
                }
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    auto half_of = [&](const v4i& q) { return ((unsigned)q[e >> 1] >> ((e & 1) * 16)) & 0xffffu; };
                    to[e] = v2i{(int)(half_of(v[0]) | half_of(v[1]) << 16), (int)(half_of(v[2]) | half_of(v[3]) << 16)};
                }
            }
        }
    } else {
        for (int i = threadIdx.x; i < in_rows * p.in_w; i += 256) {
            const int r = (int)exhip_divide((unsigned)i, (unsigned)p.in_w, p.pieces_magic, p.pieces_shift), x = i - r * p.in_w, iy = iy0 + r;
            plane_t v[4] = {};
            unsigned word[4] = {};
            if ((unsigned)iy < (unsigned)p.in_h) {
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    if (c < p.in_c) v[c] = image[(size_t)c * plane + iy * p.in_w + x];
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    if (c < p.in_c) {
                        if constexpr (I8) word[c] = (unsigned)exhip_q8(scaled(v[c], c) * p.fs_in) & 0xff;
                        else word[c] = p.mean ? exhip_f2h(scaled(exhip_h2f(v[c]), c)) : v[c];
                    }
            }
            if constexpr (I8) px[r * p.row_pixels + p.pad_l + x] = (int)(word[0] | word[1] << 8 | word[2] << 16 | word[3] << 24);
            else px[r * p.row_pixels + p.pad_l + x] = v2i{(int)(word[0] | word[1] << 16), (int)(word[2] | word[3] << 16)};
        }
    }
    const int beside = p.row_pixels - p.in_w;  // padding: left of a row's pixels and behind them
    for (int r = wave; r < in_rows; r += 4)
        for (int x = lane; x < beside; x += 64) px[r * p.row_pixels + (x < p.pad_l ? x : x + p.in_w)] = pixel_t{};
    const int count = rows * p.out_w, blocks = (count + 31) / 32, items = blocks * ((p.kblocks + MT - 1) / MT);
    int b = wave, kb = 0;
    while (b >= blocks) b -= blocks, kb += MT;
    if (wave < items) load_block(kb);
    __syncthreads();
    const unsigned first = (img * (unsigned)p.out_h + (unsigned)oy0) * (unsigned)p.out_w, end = first + (unsigned)count;
    for (int item = wave; item < items; item += 4) {
        if (MT == 2 || lane < 32) {
#pragma unroll
            for (int i = 0; i < kParams; ++i) *reinterpret_cast<float*>(lds + (i * MT * 32 + lane) * 4) = par[i];
        }
        const int at = min(b * 32 + (lane & 31), count - 1);
        const int row = (int)exhip_divide((unsigned)at, (unsigned)p.out_w, p.width_magic, p.width_shift), col = at - row * p.out_w;
        const pixel_t* src = px + row * p.stride * p.row_pixels + col * p.stride + (lane >> 5) * (I8 ? 4 : 2);
        typedef typename std::conditional<I8, v16i, v16f>::type acc_t;
        acc_t acc[MT][1];
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[m][0][e] = 0;
#pragma unroll
        for (int r = 0; r < KH; ++r) {
            const pixel_t* const t = src + r * p.row_pixels;
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                if constexpr (I8) acc[m][0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[r][m], v4i{t[0], t[1], t[2], t[3]}, acc[m][0], 0, 0, 0);
                else acc[m][0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, a[r][m]), __builtin_bit_cast(v8h, v4i{t[0][0], t[0][1], t[1][0], t[1][1]}), acc[m][0], 0, 0, 0);
            }
        }
        pw_epilogue<DT, MT, 1, EP>(p, acc, first + b * 32, end, kb, lane, lds);
        b += 4;
        if (b >= blocks && item + 4 < items) {
            while (b >= blocks) b -= blocks, kb += MT;
            load_block(kb);
        }
    }
}

template <int S, int PX, bool SMALL>
int go_dw(exhip_ctx* ctx, PwParams& p) {
    // the depthwise weights, later the waves' epilogue slices; behind them the depthwise results
    p.dw_mid = std::max(4 * wave_bytes(EXHIP_F16, 1), p.xs_b / 8 * 144);
    const int lds = p.dw_mid + p.dw_pixels * (p.xs_b + 16);
    auto run = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(p.items), dim3(256), lds, ctx->stream, p);
        EXHIP_LAUNCH_CHECK();
        return 0;
    };
    const int res = !p.residual ? 0 : p.residual_last ? 2 : 1;
    if (!p.post_relu && !p.post_op && p.act == 0 && res < 2)
        return res ? run(dw_pw_kernel<S, PX, SMALL, Ep<0, kPostNone, 1>>) : run(dw_pw_kernel<S, PX, SMALL, Ep<0, kPostNone, 0>>);
    if (!p.post_relu && p.act == 0 && p.post_op == EXHIP_POST_PRELU && res == 0) return run(dw_pw_kernel<S, PX, SMALL, Ep<0, kPostPrelu, 0>>);
    return run(dw_pw_kernel<S, PX, SMALL, EpAny>);
}

template <int DT, int MT, bool VEC>
int go_stem(exhip_ctx* ctx, const PwParams& p, int lds) {
    auto run = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(p.items), dim3(256), lds, ctx->stream, p);
        EXHIP_LAUNCH_CHECK();
        return 0;
    };
    if (!p.post_op && !p.post_relu && p.act == 0) return run(stem_planes_kernel<DT, MT, VEC, Ep<0, kPostNone, 0>>);
    if (!p.post_op && !p.post_relu && p.act == 1) return run(stem_planes_kernel<DT, MT, VEC, Ep<1, kPostNone, 0>>);
    if (!p.post_op && p.post_relu && p.act == 0) return run(stem_planes_kernel<DT, MT, VEC, Ep<0, kPostRelu, 0>>);
    if constexpr (DT == EXHIP_F16)
        if (!p.post_relu && p.act == 0 && p.post_op == EXHIP_POST_PRELU) return run(stem_planes_kernel<DT, MT, VEC, Ep<0, kPostPrelu, 0>>);
    return run(stem_planes_kernel<DT, MT, VEC, EpAny>);
}

// Geometry checks and the rows of a group, shared by the two data types.
template <int DT>
int run_stem(exhip_ctx* ctx, const exhip_pw_geom& g, const exhip_pw_taps& t, int channels, PwParams& p) {
    constexpr int kSlots = DT == EXHIP_I8 ? 8 : 4, kPixelBytes = DT == EXHIP_I8 ? 4 : 8;   // a k-step's taps, a pixel in LDS
    if (g_exhip_options.stem == 0 || t.kh != 3 || t.kw > kSlots || t.stride < 1 || channels > 4 || g.k_stride % (DT == EXHIP_I8 ? 16 : 8) != 0 ||
        !pw_row_fits(4ll * g.k_stride) || g.pixels != (long long)t.n * t.out_h * t.out_w || g.pixels >= (1ll << 31) ||
        g.pixels * 4 * g.k_stride >= (1ll << 40) || (long long)t.in_h * t.in_w >= (1ll << 28))
        return EXHIP_ERR_UNSUPPORTED;
    p.in_c = channels;
    p.pixels = (unsigned)g.pixels; p.w_bytes = (unsigned)(g.slabs * t.kh * g.slab_blocks * 1024);
    p.mts = g.slab_blocks; p.K = g.k; p.kstride = g.k_stride;
    p.act = g.act; p.post_relu = g.post_relu; p.post_op = g.post_op; p.post_alpha = g.post_alpha; p.post_beta = g.post_beta;
    p.post_slope = g.post_slope; p.post_slope_shared = g.post_slope_shared;
    p.in_h = t.in_h; p.in_w = t.in_w; p.out_h = t.out_h; p.out_w = t.out_w; p.stride = t.stride; p.pad_t = t.pad_t; p.pad_l = t.pad_l;
    p.kblocks = std::min(g.slabs * g.slab_blocks, (std::max(g.k, g.k_stride) + 31) / 32);
    p.row_pixels = std::max((t.out_w - 1) * t.stride + kSlots, t.pad_l + t.in_w);
    p.row_pixels += p.row_pixels & 1;
    const int mt = p.kblocks == 1 ? 1 : 2, slices = 4 * wave_bytes(DT, mt);
    auto bytes = [&](int rows) { return slices + ((rows - 1) * t.stride + t.kh) * p.row_pixels * kPixelBytes; };
    if (bytes(1) > 65536) return EXHIP_ERR_UNSUPPORTED;
    p.tile_rows = 1;
    auto groups = [&](int rows) { return (long long)t.n * ((t.out_h + rows - 1) / rows); };
    // Rows of a group: as many as leave four groups for every CU (16 x 112 x 112 -> 64: 5.1 us with one, 5.8 with four, 7.9 with eight), up to 512
    // pixels and 32 KiB of LDS, five groups on a CU (64 x 112 x 112: 13.0 with one, 10.6 with two, 9.5 with four; 64 x 224 x 224: 29.9, 26.2, 25.9 and with
    // eight 28.7).
    if (g_exhip_options.stem > 1) p.tile_rows = std::min(g_exhip_options.stem, t.out_h);
    else while (p.tile_rows < 8 && groups(p.tile_rows * 2) >= 1024 && p.tile_rows * 2 * t.out_w <= 512 && bytes(p.tile_rows * 2) <= 32768) p.tile_rows *= 2;
    while (p.tile_rows > 1 && bytes(p.tile_rows) > 65536) --p.tile_rows;
    if (groups(p.tile_rows) >= (1ll << 31)) return EXHIP_ERR_UNSUPPORTED;
    p.items = (unsigned)groups(p.tile_rows);
    p.ch_groups = (unsigned)((t.out_h + p.tile_rows - 1) / p.tile_rows);
    exhip_host_divisor(p.ch_groups, &p.groups_magic, &p.groups_shift);
    exhip_host_divisor((unsigned)t.out_w, &p.width_magic, &p.width_shift);
    const bool vec = t.in_w % 8 == 0 && (uintptr_t)p.x % 16 == 0;
    p.pieces = t.in_w / 8;
    exhip_host_divisor((unsigned)(vec ? p.pieces : t.in_w), &p.pieces_magic, &p.pieces_shift);
    const int lds = bytes(p.tile_rows);
    if (mt == 1) return vec ? go_stem<DT, 1, true>(ctx, p, lds) : go_stem<DT, 1, false>(ctx, p, lds);
    return vec ? go_stem<DT, 2, true>(ctx, p, lds) : go_stem<DT, 2, false>(ctx, p, lds);
}

thread_local exhip_waiting<PwParams>* t_collect = nullptr;  // (exhip_pw_pair)

// U > 0: the kernel with U k-steps a request round, 100 + U in pairs; U < 0: the split form, -kSplit a k-step at a time, -2 * kSplit in pairs
template <int DT, int MT, int NT, int U, bool TAPS, typename EP>
int go(exhip_ctx* ctx, const PwParams& p) {
    if constexpr (two_kind<DT, MT, NT, U, TAPS, EP>() >= 0) {
        if (t_collect) {
            t_collect->kind = two_kind<DT, MT, NT, U, TAPS, EP>();
            t_collect->dt = DT;
            t_collect->groups = U < 0 ? p.items : (p.items + 3) / 4;
            if constexpr (U < 0) t_collect->kernel = reinterpret_cast<const void*>(conv_pw_split_kernel<DT, MT, kSplit, TAPS, U == -2 * kSplit, EP>);
            else t_collect->kernel = reinterpret_cast<const void*>(conv1x1_pw_kernel<DT, MT, NT, U % 100, TAPS, (U > 100), EP>);
            t_collect->p = p;
            t_collect = nullptr;
            return 0;
        }
    }
    if constexpr (U < 0) hipLaunchKernelGGL((conv_pw_split_kernel<DT, MT, kSplit, TAPS, U == -2 * kSplit, EP>), dim3(p.items), dim3(64 * kSplit), 0, ctx->stream, p);
    else hipLaunchKernelGGL((conv1x1_pw_kernel<DT, MT, NT, U % 100, TAPS, (U > 100), EP>), dim3((p.items + 3) / 4), dim3(256), 0, ctx->stream, p);
    EXHIP_LAUNCH_CHECK();
    return 0;
}

// The layers behind the convolution, as template constants where a network of this library's kind has the combination.
template <int DT, int MT, int NT, int U, bool TAPS>
int pick_epilogue(exhip_ctx* ctx, const PwParams& p) {
    const bool shortcut = DT == EXHIP_I8 ? p.residual_f != nullptr : p.residual != nullptr;
    const int res = !shortcut ? 0 : p.residual_last ? 2 : 1;
    int post = p.post_relu ? kPostRelu : kPostNone;
    if (p.post_op) {
        const int op = p.post_op == EXHIP_POST_PRELU ? kPostPrelu
                       : p.post_op == 1 + EXHIP_UNARY_HARDSWISH ? kPostHardSwish
                       : p.post_op == 1 + EXHIP_UNARY_LEAKYRELU ? kPostLeaky : -1;
        post = post == kPostNone ? op : -1;
    }
    const bool bn = p.post_bn_a != nullptr;
    if (p.pool) {
        if constexpr (DT == EXHIP_I8 && TAPS && U > 0) {
            if (p.act == 0 && post == kPostNone) return go<DT, MT, NT, U, TAPS, Pooled<Ep<0, kPostNone, 0>>>(ctx, p);
            if (p.act == 0 && post == kPostRelu) return go<DT, MT, NT, U, TAPS, Pooled<Ep<0, kPostRelu, 0>>>(ctx, p);
            if (p.act == 1 && post == kPostNone) return go<DT, MT, NT, U, TAPS, Pooled<Ep<1, kPostNone, 0>>>(ctx, p);
        }
        return EXHIP_ERR_UNSUPPORTED;
    }
    if (p.group) return go<DT, MT, NT, U == 8 ? 4 : U, TAPS, EpAny>(ctx, p);
    auto is = [&](int a, int q, int r, bool b) { return p.act == a && post == q && res == r && bn == b; };
    if (is(0, kPostNone, 0, false)) return go<DT, MT, NT, U, TAPS, Ep<0, kPostNone, 0>>(ctx, p);
    if (is(0, kPostHardSwish, 0, false)) return go<DT, MT, NT, U, TAPS, Ep<0, kPostHardSwish, 0>>(ctx, p);
    if (is(0, kPostRelu, 0, false)) return go<DT, MT, NT, U, TAPS, Ep<0, kPostRelu, 0>>(ctx, p);
    if (is(1, kPostNone, 0, false)) return go<DT, MT, NT, U, TAPS, Ep<1, kPostNone, 0>>(ctx, p);
    if (is(0, kPostHardSwish, 2, false)) return go<DT, MT, NT, U, TAPS, Ep<0, kPostHardSwish, 2>>(ctx, p);
    if (is(0, kPostRelu, 1, false)) return go<DT, MT, NT, U, TAPS, Ep<0, kPostRelu, 1>>(ctx, p);
    if constexpr (DT == EXHIP_F16) {
        if (is(0, kPostPrelu, 0, false)) return go<DT, MT, NT, U, TAPS, Ep<0, kPostPrelu, 0>>(ctx, p);
        if (is(0, kPostNone, 1, false)) return go<DT, MT, NT, U, TAPS, Ep<0, kPostNone, 1>>(ctx, p);
    } else {
        if (is(0, kPostRelu, 2, false)) return go<DT, MT, NT, U, TAPS, Ep<0, kPostRelu, 2>>(ctx, p);
        if constexpr (!TAPS)
            if (is(0, kPostLeaky, 0, true)) return go<DT, MT, NT, U, TAPS, Ep<0, kPostLeaky, 0, true>>(ctx, p);
    }
    return go<DT, MT, NT, U == 8 ? 4 : U, TAPS, EpAny>(ctx, p);
}

// Whether a launch takes the split form: long enough reductions, few enough blocks of 32 pixels x 32 channels. Its waves request their
// pixels in 64-byte pieces (`pairs`), which the other kernels for these layers do not, so it also wins where every SIMD has several
// waves. Measured over 64 to 1024 channels on maps of 20, 40 and 80 at 1 to 32 images, us without -> with it; a line lies between
// the largest launch that wins throughout and the next one measured:
//  * 1x1, from 16 k-steps on: fp16 800 blocks 5.7 -> 4.2, 1600 6.1 -> 5.8, 6400 15.5 -> 14.0 (64 k-steps 13.6 -> 6.7, 14.3 -> 10.6,
//    48 -> 31); int8 32 k-steps 3200 blocks 15.1 -> 11.5 (6400 20.5
//    against 20.9), 16 k-steps 800 blocks 6.1 -> 4.6 (1600 6.30 against 6.40).
//    8 k-steps: fp16 800 blocks 4.19 -> 4.05, 1600 4.5 against 5.1; int8 800 blocks 4.55 against 4.9.
//  * a filter at stride 1, against the lean kernel: 1200 blocks fp16 9.2 -> 7.3 (36 k-steps), 12.8 -> 10.6 (72), 19.7 -> 18.0
//    (144), int8 6.05 -> 4.95 (18), 9.7 -> 7.4 (36); 1600 blocks fp16 12.5 against 13.3 (72), int8 6.2 against 6.7 (18), 11.5 against
//    13.4 (72, but 20.3 -> 13.3 with an activation layer behind, 2400 blocks 21.1 -> 16.9, 3200 21.5 against 22.3).
//  * a filter at stride 2, against the tapped form: int8 1600 blocks 6.3 against 6.9 (18), 8.6 against 9.4 (36), fp16 3200 blocks 12.3
//    against 14.1 (36), 20.0 against 24.5 (72); beyond the tapped form's k-steps against the staged kernel: 1600 blocks 30.7 -> 23.7
//    (fp16, 144) and 28.6 -> 23.8 (int8, 144), 3200 blocks 38 and 35 against 42.
// Layers without pairs (32-byte pixels, an odd number of chunks): 800 blocks. A lone 32-channel block would leave half of every tile
// unused.
bool split_wins(int dt, const exhip_pw_geom& g, int kblocks, int n_ksteps, bool taps, int stride) {
    if (g_exhip_options.force_splits == 1 || g_exhip_options.pw_split == 0 || kblocks < 2) return false;
    if (g_exhip_options.pw_split == 2) return true;
    if (n_ksteps < 8) return false;
    const long long blocks = (g.pixels + 31) / 32 * kblocks;
    if (g.c_bytes % 64 != 0) return blocks <= 832;
    if (!taps) {
        if (dt == EXHIP_I8) return blocks <= (n_ksteps < 16 ? 640 : n_ksteps < 32 ? 832 : 3328);
        return blocks <= (n_ksteps < 16 ? 832 : 6656);
    }
    if (stride != 1) return blocks <= (n_ksteps < 16 ? 832 : n_ksteps < 64 ? (dt == EXHIP_I8 ? 1280 : 1920) : blocks * n_ksteps <= 240000 ? 1920 : 832);
    // (parts of blocks, and more k-steps than the tapped form takes, leave the staged kernel: int8 384 -> 48 at 1600 blocks 23.5 -> 18.6)
    if (dt == EXHIP_I8 && n_ksteps > 2 * kMaxDirectSteps && g.k % 32 != 0 && !g.post_op) return blocks <= 1664;
    if (dt == EXHIP_I8 && n_ksteps >= 64 && g.post_op) {
        // beyond 100 k-steps, of whole blocks, the products decide: up to 1216 tiles (384 -> 64 at 1000 tiles 19.9 and 19.7, at 1231 20.0 against 23.2, 384 -> 96 at
        // 1184 24.2 -> 22.4, at 1432 24.0 against 26.8)
        const long long tiles = (g.pixels + 31) / 32 * ((kblocks + 1) / 2);
        return blocks <= 2560 && (n_ksteps <= 100 || g.k % 32 != 0 || tiles <= 1216);
    }
    return blocks <= 1280;
}

// Where a pixel's bytes of a tap (of all channels for a 1x1 layer) come in whole 64-byte pieces, the k-steps are taken in pairs. A
// packing in chunks of 32 bytes gives them too if the chunks are even in number: a pair's second k-step is the next chunk's then
// (`any_order`: unsplit fp16 sums keep the order of the general kernel's, and so its bits).
template <bool TAPS>
bool plan_pairs(PwParams& p, bool any_order) {
    const int taps = TAPS ? p.kh * p.kw : 1;
    const bool two_chunks = TAPS && p.chunk_b == 32 && any_order && p.n_ksteps / taps % 2 == 0;
    const bool pairs = two_chunks || (TAPS ? p.chunk_b : p.n_ksteps * 32) % 64 == 0;
    if (two_chunks) {
        p.chunk_end_b += 32;
        p.chunk_b = 64;
    }
    p.pair_w = two_chunks ? taps : 1;
    p.next_w = two_chunks ? 1 : 2;
    p.chunk_w = two_chunks ? taps : 0;
    return pairs;
}

template <int DT, int MT, int NT, bool TAPS = false>
int launch(exhip_ctx* ctx, PwParams& p, int kblocks) {
    // (two k-steps and no filter: pixels of 64 bytes, which lie side by side in the tensor: 64 -> 32 at 16 x 160 x 160 int8 9.6, in pairs 9.8)
    const bool pairs = MT + NT <= 3 && (TAPS || p.n_ksteps >= 4) && plan_pairs<TAPS>(p, DT == EXHIP_I8);
    if (TAPS) {
        const int taps = p.kh * p.kw, per_tap = p.chunk_b / 32;
        const int each = pairs ? 2 : 1;
        if (p.n_ksteps > each * kMaxDirectSteps) return EXHIP_ERR_UNSUPPORTED;
        for (int i = 0; i * each < p.n_ksteps; ++i) {
            const int s = i * each, chunk = s / (taps * per_tap), tap = s / per_tap % taps, r = tap / p.kw, q = tap % p.kw;
            p.step[i] = ((r * p.in_w + q) * p.xs_b + chunk * p.chunk_b + s % per_tap * 32) | (int)((unsigned)tap << kTapShift);
            p.pair_first[i] = pairs && p.next_w == 1 ? chunk * 2 * taps + tap : s;
        }
    }
    const long long tiles = ((long long)p.pixels + 32 * NT - 1) / (32 * NT);
    p.ch_groups = (unsigned)((kblocks + MT - 1) / MT);
    const long long items = tiles * p.ch_groups;
    if (items >= (1ll << 31) - 4) return EXHIP_ERR_UNSUPPORTED;
    p.items = (unsigned)items;
    exhip_host_divisor(p.ch_groups, &p.groups_magic, &p.groups_shift);
    if constexpr (MT + NT > 3) {
        return go<DT, MT, NT, 2, TAPS, EpAny>(ctx, p);
    } else {
        if (pairs) return pick_epilogue<DT, MT, NT, 104, TAPS>(ctx, p);
        // A launch of at most two waves per SIMD is as long as one wave's chain of load round trips: sixteen k-steps in flight
        // where there are more than eight. Larger ones hide each other's round trips and want the registers for more waves.
        if constexpr (MT == 2)
            if (items <= 2048 && p.n_ksteps > 8) return pick_epilogue<DT, MT, NT, 8, TAPS>(ctx, p);
        return pick_epilogue<DT, MT, NT, 4, TAPS>(ctx, p);
    }
}

// The k-step where wave i of a split tile begins.
int split_start(int n_ksteps, bool pairs, int i) {
    return pairs ? (int)((long long)(n_ksteps / 2) * i / kSplit) * 2 : (int)((long long)n_ksteps * i / kSplit);
}

template <int DT, bool TAPS>
int launch_split(exhip_ctx* ctx, PwParams& p, int kblocks) {
    p.ch_groups = (unsigned)((kblocks + 1) / 2);
    const long long items = ((long long)p.pixels + 31) / 32 * p.ch_groups;
    if (items >= (1ll << 31) - 4) return EXHIP_ERR_UNSUPPORTED;
    p.items = (unsigned)items;
    exhip_host_divisor(p.ch_groups, &p.groups_magic, &p.groups_shift);
    const bool pairs = plan_pairs<TAPS>(p, true), two_chunks = pairs && p.next_w == 1;
    for (int i = 0; i <= kSplit; ++i) {
        const int s = split_start(p.n_ksteps, pairs, i);
        p.start_s[i] = s;
        p.start_w[i] = s;
        if (TAPS) {
            const int per_tap = p.chunk_b / 32, per_row = p.kw * per_tap, per_chunk = p.kh * per_row;
            const int chunk = s / per_chunk, in_chunk = s % per_chunk, row = in_chunk / per_row, tap = in_chunk % per_row / per_tap, k = in_chunk % per_tap;
            if (two_chunks) p.start_w[i] = chunk * per_chunk + in_chunk / 2;
            p.start_r[i] = row;
            p.start_q[i] = tap;
            p.start_b[i] = (row * p.in_w + tap) * p.xs_b + chunk * p.chunk_b + k * 32;
            p.start_left[i] = p.chunk_b - k * 32;
        }
    }
    return pairs ? pick_epilogue<DT, 2, 1, -2 * kSplit, TAPS>(ctx, p) : pick_epilogue<DT, 2, 1, -kSplit, TAPS>(ctx, p);
}

}  // namespace

namespace {

// Layers of more than 32 output channels take the 32-pixel x 64-channel wave tile whatever their size: half the registers of
// the 64 x 64 tile, so more waves hide each other's loads and epilogues. Measured on whole forwards against "64 x 64 from
// 2048 waves on" (option pw_tile = 2): int8 64 -> 64 at 16 x 160 x 160 41 -> 30 us, a detection network's int8 forward
// 1.44 -> 1.35 ms, its fp16 forward 1.81 -> 1.79 ms, two mobile networks' fp16 forwards 0.435 -> 0.42 and 0.82 -> 0.805 ms.
template <int DT>
bool small_tile() { return g_exhip_options.pw_tile != 2; }

// A layer with a filter, a stride or padding on the same kernel: g.pixels counts output pixels, the k-steps walk the
// packing's order (channel chunk, filter row, tap, 32-byte step).
template <int DT>
int run_taps(exhip_ctx* ctx, const exhip_pw_geom& g, const exhip_pw_taps& t, PwParams& p, bool has_residual) {
    if (g_exhip_options.direct == 0) return EXHIP_ERR_UNSUPPORTED;
    if (g.post_bn_a || g.post_bn_b || g.exact_k || g.group) return EXHIP_ERR_UNSUPPORTED;
    if (g.pool && (DT != EXHIP_I8 || has_residual || t.out_h % 2 || t.out_w % 2)) return EXHIP_ERR_UNSUPPORTED;
    const long long n_ksteps = (long long)t.n_chunks * t.kh * t.kw * (t.chunk_b / 32);
    if (g.pixels <= 0 || g.c_bytes <= 0 || g.c_bytes % 32 != 0 || t.chunk_b % 32 != 0 || t.n_chunks * t.chunk_b != g.c_bytes ||
        (g.slab_blocks != 2 && g.slab_blocks != 4) || g.k_stride % 8 != 0 || !pw_row_fits(4ll * g.k_stride) || t.kh * t.kw > (1 << (32 - kTapShift)) || t.stride < 1 || t.pad_t < 0 || t.pad_l < 0)
        return EXHIP_ERR_UNSUPPORTED;
    const long long x_bytes = (long long)t.n * t.in_h * t.in_w * g.c_bytes;
    const long long w_bytes = (long long)g.slabs * n_ksteps * g.slab_blocks * 1024;
    const long long reach = ((long long)(t.kh - 1) * t.in_w + t.kw) * g.c_bytes;   // the furthest step behind a pixel's top-left tap
    if (x_bytes >= kOutOfRange || w_bytes >= kOutOfRange || reach >= (1ll << kTapShift) || g.pixels != (long long)t.n * t.out_h * t.out_w ||
        g.pixels * 4 * g.k_stride >= (1ll << 40) || g.pixels >= (1ll << 31))
        return EXHIP_ERR_UNSUPPORTED;
    if (g.post_op && g.post_op != EXHIP_POST_PRELU && (g.post_op < 1 || g.post_op > 1 + EXHIP_UNARY_CLIP || g.post_op == 1 + EXHIP_UNARY_SIGMOID))
        return EXHIP_ERR_UNSUPPORTED;
    const int kblocks = std::min(g.slabs * g.slab_blocks, (std::max(g.k, g.k_stride) + 31) / 32);
    p.post_slope = g.post_slope;
    p.pixels = (unsigned)g.pixels; p.x_bytes = (unsigned)x_bytes; p.w_bytes = (unsigned)w_bytes;
    p.xs_b = g.c_bytes; p.n_ksteps = (int)n_ksteps; p.mts = g.slab_blocks;
    p.K = g.k; p.kstride = g.k_stride;
    p.act = g.act; p.post_relu = g.post_relu; p.post_op = g.post_op; p.post_slope_shared = g.post_slope_shared;
    p.residual_last = g.residual_last && has_residual;
    p.post_alpha = g.post_alpha; p.post_beta = g.post_beta;
    p.pool = g.pool;
    p.in_h = t.in_h; p.in_w = t.in_w; p.out_h = t.out_h >> g.pool; p.out_w = t.out_w >> g.pool; p.stride = t.stride; p.pad_t = t.pad_t; p.pad_l = t.pad_l;
    p.kh = t.kh; p.kw = t.kw;
    exhip_host_divisor((unsigned)(p.out_h * p.out_w), &p.image_magic, &p.image_shift);
    exhip_host_divisor((unsigned)p.out_w, &p.width_magic, &p.width_shift);
    p.chunk_b = t.chunk_b;
    p.row_end_b = (t.in_w - t.kw) * g.c_bytes;
    p.chunk_end_b = t.chunk_b - t.kh * t.in_w * g.c_bytes;
    if (t.staged) return exhip_conv3x3_staged(ctx, DT, &p, t.n, kblocks, t.lean_tiles);
    if (n_ksteps > (g.c_bytes % 64 ? 1 : 2) * kMaxDirectSteps && !split_wins(DT, g, kblocks, (int)n_ksteps, true, t.stride)) return EXHIP_ERR_UNSUPPORTED;
    // Every fp16 layer that the lean kernel leaves (stride 2, 12 or 32 input channels, ragged output channels): 128 -> 256 3x3 at stride
    // 2 from 16 x 80 x 80 48.6 us on the staged kernel, 36.9 here; 64 -> 128 from 16 x 160 x 160 71.9 and 35.8. A lone 32-channel block and
    // 32-byte pixels win whatever their size (12 -> 32 at 16 x 320 x 320 int8 71 -> 46 us, 32 -> 32 at 16 x 160 x 160 24.9 -> 15.8).
    // Other int8 layers by what stands behind the products, us on the staged or lean kernel -> here, over some 60 maps from 16 to 111 wide:
    //  * stride 2: everything, 27.5 -> 21.9 (256 -> 256 at 48 x 37 x 34), 17.4 -> 11.1 with a float32 result (64 -> 128 at 48 x 50 x 47) --
    //    but with an int8 result alone large maps in powers of two stay (128 -> 256 at 16 x 80 x 80 17.1 against 21.5): up to 4800
    //    blocks of 32 x 32 (17.9 -> 16.8) and three waves a SIMD (192 -> 96 at 8 x 80 x 80, 3200 waves, 24.9 against 28.9). A ReLU alone behind
    //    whole blocks makes the staged kernel faster (192 -> 96 at stride 1, 2 x 106 x 109, 13.1 with it, 16.2 without): two waves a SIMD there beyond 40
    //    k-steps or without pairs (256 -> 96 at 5 x 80 x 80, 2000 waves, 24.4 -> 20.9, at 7 x 75 x 75, 2462 waves, 26.0 against 28.9).
    //  * stride 1, where the lean kernel takes a plain ReLU in 8.7 us for 128 -> 128 at 16 x 40 x 40 and this one in 12.2: an activation
    //    layer (17.8 -> 12.0; 64 -> 64 at 8 x 80 x 80 9.9 -> 8.1, at 16 x 80 x 80 12.2 against 13.4), a float32 result beside the
    //    int8 one (20.9 -> 14.6 at 4 x 80 x 80, 40.5 -> 40.2 at 11 856 blocks; 72 k-steps 27.9 -> 23.6 at 4096, 37.1 against 40.4 at
    //    6400; 18 k-steps but for 5632 to 8192 blocks, one full round of the lean kernel, 14.4 against 15.7 at 6400), no activation at all, which the
    //    lean kernel has no form for (18 k-steps 9.7 -> 6.4 at 1600, 11.1 -> 9.8 at 4800, 11.5 against 12.5 at 6400; 36 16.0 -> 8.5 and 22.7 -> 19.1 at 6400,
    //    17.3 against 19.2 at 7504; 72 20.5 -> 18.7 at 3200, 18.3 against 18.8 at 3752), a sum (17.6 -> 15.3 at 3200, 20.8 against 21.4 at 4376; 18 k-steps 8.8 -> 8.4 at 1944, 9.2 against 10.8 at 2376; 72 never),
    //    the ReLU behind (13.7 -> 12.2; 18 k-steps never).
    const long long blocks = (g.pixels + 31) / 32 * kblocks, waves = kblocks == 1 ? (g.pixels + 63) / 64 : (g.pixels + 31) / 32 * ((kblocks + 1) / 2);
    const bool relu_alone = DT == EXHIP_I8 && (g.act == 1 || g.post_relu) && g.k % 32 == 0 && !g.post_op && !has_residual && !p.y_f;
    auto int8_most = [&]() -> long long {
        const long long all = 1ll << 40;
        if (t.stride != 1) return g.post_op || has_residual || p.y_f ? all : waves <= (relu_alone && (n_ksteps > 40 || g.c_bytes % 64 != 0) ? 2048 : 3072) ? 4800 : 0;
        if (t.kh != 3 || t.kw != 3 || t.chunk_b != 64 || g.k % 64 != 0) return 3328;  // the staged kernel's
        if (g.post_op) return n_ksteps <= 40 ? 4096 : 3328;
        if (has_residual) return n_ksteps <= 18 ? 2048 : n_ksteps <= 40 ? 3328 : 0;
        if (p.y_f) return n_ksteps <= 18 && blocks > 5632 && blocks <= 8192 ? 0 : n_ksteps <= 40 ? 12000 : 4096;
        if (!g.act && !g.post_relu) return n_ksteps <= 18 ? 4800 : n_ksteps <= 40 ? 6400 : 3328;
        return g.post_relu && n_ksteps > 18 ? 3328 : 0;
    };
    // Layers at stride 1 of more than 40 k-steps and ragged output channels once more go to the staged kernel from the second round of waves on
    // (two a SIMD): fp16 96 -> 96 at 5 x 80 x 80 (2000 waves) 16.7 -> 14.9, at 8 x 80 x 80 (3200) 19.9 against 24.7, 128 -> 205 at 3 x 102 x 101
    // 25.1 against 34.1. A lone block's waves have 64 pixels: fp16 96 -> 32 at 16 x 80 x 80 (1600) 17.6 -> 17.1, at 29 x 69 x 69 (2158) 23.2 against
    // 26.6; int8 192 -> 32 at 23 x 52 x 52 (972) 16.5 -> 12.2, at 17 x 71 x 71 (1340) 15.9 against 16.6, 256 -> 32 at 24 x 83 x 82 29.2 against 34.9.
    // The figures are us on the staged kernel -> here. int8 layers with a ReLU alone (above): from the second wave a SIMD on (192 -> 96 at 2 x 80 x 80, 800
    // waves, 14.5 -> 10.9, at 3 x 75 x 75, 1056 waves, 13.3 against 14.3), and a lone block of 72 k-steps on fewer than one SIMD in four, which the staged
    // kernel splits (256 -> 32 at 1 x 80 x 80 12.6 against 14.0, at 28 x 26 x 26, 296 waves, 14.8 -> 14.3).
    const bool late = t.stride == 1 && n_ksteps > 40 && g.k % 64 != 0 &&
                      (waves > (relu_alone ? 1024 : kblocks > 1 ? 2048 : DT == EXHIP_F16 ? 1664 : 1024) || (relu_alone && kblocks == 1 && n_ksteps >= 64 && waves <= 256));
    const bool take = g.pool || g.c_bytes == 32 || (!late && (kblocks == 1 || DT == EXHIP_F16 || blocks <= int8_most()));
    // With the pooling layer behind it: where the layer by itself would run in the split form, on few blocks, that and a launch for the pooling are
    // the faster two, us as two launches -> as one: 64 -> 128 at 1 x 30 x 30 7.4 -> 6.4, 128 -> 128 at 1 x 14 x 14 (36 k-steps) 8.0 against 8.4, at 16
    // x 14 x 14 (288 blocks) 8.7 and 8.6, 256 -> 256 at 4 x 16 x 16 (72 k-steps) 9.5 against 13.2, at 16 x 16 x 16 (1024) 14.2 -> 13.5. Beyond, the float32
    // map that is neither stored nor read decides: 32 -> 64 at 64 x 62 x 62 31.6 -> 17.2, 64 -> 64 at 64 x 112 x 112 112.9 -> 64.2.
    if (g.pool && g_exhip_options.direct != 2 && blocks <= (n_ksteps <= 18 ? 0 : n_ksteps <= 40 ? 300 : 960)) return EXHIP_ERR_UNSUPPORTED;
    const bool split = !g.pool && split_wins(DT, g, kblocks, (int)n_ksteps, true, t.stride);
    if (g_exhip_options.direct != 2 && !take && !split) return EXHIP_ERR_UNSUPPORTED;
    if (split) return launch_split<DT, true>(ctx, p, kblocks);
    if (kblocks == 1) return launch<DT, 1, 2, true>(ctx, p, kblocks);
    // (the 64 x 64 tile has no pooled epilogue: its kernel would take the convolution's pixels, four times as many, for the pooled map's)
    const long long waves64 = ((g.pixels + 63) / 64) * ((kblocks + 1) / 2);
    if (g.pool || waves64 < 2048 || small_tile<DT>()) return launch<DT, 2, 1, true>(ctx, p, kblocks);
    return launch<DT, 2, 2, true>(ctx, p, kblocks);
}

// The pointwise layer p behind the depthwise layer dw.
int run_depthwise(exhip_ctx* ctx, const exhip_pw_depthwise& dw, PwParams& p, int kblocks, bool split) {
    if (g_exhip_options.dw_pw == 0) return EXHIP_ERR_UNSUPPORTED;
    const long long x_bytes = (long long)dw.n * dw.in_h * dw.in_w * p.xs_b;
    if (p.xs_b > 1024 || x_bytes > (1ll << 30) || (dw.stride != 1 && dw.stride != 2) || (dw.act != 0 && dw.act != 1 && dw.act != 3) ||
        (long long)dw.n * dw.out_h * dw.out_w != (long long)p.pixels)
        return EXHIP_ERR_UNSUPPORTED;
    p.x = reinterpret_cast<const char*>(dw.x); p.x_bytes = (unsigned)x_bytes;
    p.in_h = dw.in_h; p.in_w = dw.in_w; p.out_h = dw.out_h; p.out_w = dw.out_w; p.stride = dw.stride; p.pad_t = dw.pad_t; p.pad_l = dw.pad_l;
    p.dw_w = dw.w9; p.dw_bias = dw.bias; p.dw_slope = dw.slope; p.dw_slope_shared = dw.slope_shared; p.dw_act = dw.act;
    exhip_host_divisor((unsigned)(dw.out_h * dw.out_w), &p.image_magic, &p.image_shift);
    exhip_host_divisor((unsigned)dw.out_w, &p.width_magic, &p.width_shift);
    const long long tiles32 = ((long long)p.pixels + 31) / 32;
    const int widest = dw.stride == 2 ? 2 - dw.out_w % 2 : dw.out_w % 4 == 0 ? 4 : 2 - dw.out_w % 2, channels4 = p.xs_b >> 3;
    p.kblocks = kblocks;
    p.dw_split = split;
    for (int i = 0; i <= kSplit; ++i) p.start_s[i] = split_start(p.n_ksteps, p.n_ksteps % 2 == 0, i);
    // Pixels of a group. A small launch is as long as one group's chain, a strip of four channels that a thread computes behind another
    // 0.8 us of it: while the chip has room, groups of half the pixels (256 -> 128 at 1 x 14 x 14: 8.0 us with 32 pixels, 6.5 with
    // 16, 5.5 with 8, 5.2 with 4; 512 -> 128 at 1 x 7 x 7: 14.6, 10.1, 8.2, 7.1), but a second round of groups costs what
    // it saves (256 -> 128 at 16 x 14 x 14: 8.3 with 32, 6.6 with 16 in 196 groups, 6.8 with 8 in 392) unless the strips are many (512 ->
    // 128 at 64 x 7 x 7: 10.5 with 16, 9.8 with 8 in 392; 384 -> 128 at stride 2 to 305 x 32 pixels 19.1 with 32, 15.1 with 16 in 610). A large
    // launch wants a strip for every thread and no more, and two groups for every CU or so, more where many output channels follow (16 -> 256 at
    // 1182 x 32 pixels 13.8 with 256, 9.8 with 64, 9.5 with 32; 96 -> 512 at 1425 x 32 31.9 with 128, 22.5 with 64): 16 -> 32 at
    // 64 x 112 x 112 24.5 us with 256 pixels, 33.6 with 128, 55.5 with 64; 32 -> 64 43.7 with 128, 61.8 with 64; 128 -> 64 at 64 x 56 x 56
    // 33.8 with 64, 39.3 with 32; 256 -> 128 at 64 x 28 x 28 27.7 with 64, 22.7 with 32.
    p.dw_pixels = 32;
    if (tiles32 >= 1024)
        while (p.dw_pixels < 256 && p.dw_pixels * channels4 < (channels4 < 24 ? 1024 : 2048) && p.pixels / (2 * p.dw_pixels) >= (kblocks < 4 ? 448u : 640u)) p.dw_pixels *= 2;
    auto more = [&]() { return ((long long)p.pixels * 2 + p.dw_pixels - 1) / p.dw_pixels * ((kblocks + 3) / 4); };  // groups with half the pixels each
    while (p.dw_pixels > 4 && p.dw_pixels * channels4 > 256 && more() <= (p.dw_pixels * channels4 > 1024 ? 704 : 256)) p.dw_pixels /= 2;
    if (const int forced = g_exhip_options.dw_pw; forced >= 4 && forced <= 256 && (forced & (forced - 1)) == 0 && forced * (p.xs_b + 16) <= 40960) p.dw_pixels = forced;
    const bool small = p.dw_pixels < 32;
    // One launch is the faster one but for wide layers of a middling size, whose groups are few and long: 512 -> 512 at 20 x 14 x 14 16.6 us,
    // 15.8 as two launches, 384 -> 384 at 8 x 14 x 14 10.8 and 9.9, 256 -> 512 at stride 2 from 8 x 28 x 28 8.2 and 7.8; on the other
    // sides 512 -> 512 at 1 x 14 x 14 6.8 and 8.9, at 64 x 14 x 14 27.0 and 31.0, 512 -> 128 at 64 x 7 x 7 10.1 and 10.5.
    // The depthwise half reads a strip's neighbours once for all its pixels; strips of one pixel (an odd width) or two make it the longer one where a
    // launch has many: us for the pair and for the two, 384 -> 256 at 302 x 32 pixels 20.2 and 14.6, 512 -> 64 at 24 x 39 x 39 38.5 and 30.7, 192 -> 32 at 17 x 125 x 125
    // 74.4 and 57.0, 96 -> 128 at 10747 x 32 65.8 and 52.3; in strips of two 384 -> 64 at 3 x 111 x 114 28.1 and 24.8. (384 -> 96 at 885 x 32 23.3 and 27.0.)
    if (g_exhip_options.dw_pw == 1) {
        if (tiles32 > 40 && tiles32 <= 256 && kblocks > (p.xs_b > 512 ? 4 : 8)) return EXHIP_ERR_UNSUPPORTED;
        if (tiles32 > 20 && tiles32 <= 40 && kblocks > 8 && p.xs_b >= 768) return EXHIP_ERR_UNSUPPORTED;  // 384 -> 512 at 34 x 32 11.3 and 8.3
        if (widest == 1 && p.xs_b >= 768 && ((tiles32 > 256 && tiles32 <= 640) || tiles32 > (p.xs_b < 1024 ? 1024 : 768))) return EXHIP_ERR_UNSUPPORTED;
        if (widest == 1 && ((p.xs_b >= 384 && tiles32 > 2048) || (p.xs_b >= 128 && tiles32 > 6144))) return EXHIP_ERR_UNSUPPORTED;
        if (widest == 2 && p.xs_b >= 768 && tiles32 > 1024) return EXHIP_ERR_UNSUPPORTED;
    }
    p.dw_tiles = std::max(p.dw_pixels / 32, 1);
    const long long tiles = ((long long)p.pixels + p.dw_pixels - 1) / p.dw_pixels;
    int groups = 1;
    while (groups * 4 < kblocks * p.dw_tiles && tiles * groups * 2 <= 512) groups *= 2;
    p.dw_kblocks = (kblocks + groups - 1) / groups;
    p.ch_groups = (unsigned)((kblocks + p.dw_kblocks - 1) / p.dw_kblocks);
    p.items = (unsigned)(tiles * p.ch_groups);
    exhip_host_divisor(p.ch_groups, &p.groups_magic, &p.groups_shift);
    if (small) {
        int px = 1;
        while (px < widest && p.dw_pixels * channels4 / px > 256) px *= 2;
        if (dw.stride == 2) return px == 2 ? go_dw<2, 2, true>(ctx, p) : go_dw<2, 1, true>(ctx, p);
        return px == 4 ? go_dw<1, 4, true>(ctx, p) : px == 2 ? go_dw<1, 2, true>(ctx, p) : go_dw<1, 1, true>(ctx, p);
    }
    if (dw.stride == 2) return widest == 2 ? go_dw<2, 2, false>(ctx, p) : go_dw<2, 1, false>(ctx, p);
    return widest == 4 ? go_dw<1, 4, false>(ctx, p) : widest == 2 ? go_dw<1, 2, false>(ctx, p) : go_dw<1, 1, false>(ctx, p);
}

// Geometry checks and the wave tile, shared by the two data types. `es`: bytes per input element.
template <int DT>
int run_pw(exhip_ctx* ctx, const exhip_pw_geom& g, PwParams& p, int es, bool has_residual, const exhip_pw_taps* t = nullptr, const exhip_pw_depthwise* dw = nullptr) {
    if (g_exhip_options.pw == 0 || (dw && (t || g.post_bn_a || g.exact_k || g.group))) return EXHIP_ERR_UNSUPPORTED;
    if (t) return run_taps<DT>(ctx, g, *t, p, has_residual);
    // Measured per layer against the general kernel inside a detection and two mobile networks (16 and 64 images, kernel
    // traces): this form wins where a launch is short -- every layer of at most 32 768 pixels up to about 7 GFLOP (twice
    // as fast on 20 x 20 maps) --, for a lone 32-channel block (which the general kernel pads to a 64-channel slab), and on
    // larger maps while the input is narrow: fp16 up to 64 input channels (64 -> 64 at 16 x 160 x 160: 42 against 49 us)
    // and 128 -> 64 at 80 x 80; int8 up to 64 channels at 131 072 pixels, and layers with only a float32 result (its
    // 64-byte store runs against the general epilogue's 16-byte pieces: 41 against 60 us on a 128 -> 255 head at
    // 16 x 80 x 80). Beyond that the general kernel's staged tiles re-read less and win (128 -> 128 at 80 x 80).
    // Option pw = 2 takes every layer the kernel can (tests), 0 none.
    const bool joined = g.post_bn_a || g.exact_k || g.group;  // only this kernel has those: it takes the layer whatever its size
    if (joined && ((g.post_bn_a == nullptr) != (g.post_bn_b == nullptr) || (g.post_bn_a && g.post_op == EXHIP_POST_PRELU) || (g.exact_k && g.k % 32 != 0)))
        return EXHIP_ERR_UNSUPPORTED;
    if (g.group) {
        if (g.group < 0 || g.k % g.group != 0 || g.pixels % ((long long)g.map_h * g.map_w) != 0 || g.pixels * g.k >= (1ll << 32) || p.y_q || has_residual)
            return EXHIP_ERR_UNSUPPORTED;
        p.group = g.group;
        p.out_h = g.map_h;
        p.out_w = g.map_w;
        exhip_host_divisor((unsigned)(g.map_h * g.map_w), &p.image_magic, &p.image_shift);
    }
    p.post_bn_a = g.post_bn_a; p.post_bn_b = g.post_bn_b; p.exact = g.exact_k || g.group;
    const int out_channels = g.exact_k || g.group ? g.k : std::max(g.k, g.k_stride);  // channels this launch writes
    const int blocks_needed = (out_channels + 31) / 32;
    const double flop = 2.0 * (double)g.pixels * (g.c_bytes / es) * g.k;
    bool take = joined || blocks_needed == 1 || (flop <= 8.0e9 && g.pixels <= 32768);
    if (DT == EXHIP_I8 && g.pixels <= 131072 && (g.c_bytes <= 64 || (p.y_f && !p.y_q))) take = true;
    if (DT == EXHIP_I8 && g_exhip_options.pw_tile != 2 && g.c_bytes <= 512) take = true;  // with the small tile: every layer measured
    // With the small tile: every fp16 layer. Launched thirty times alone, long reductions on large maps lose a little
    // (256 -> 256 at 64 x 28 x 28: 33 against 32 us, 512 -> 512 at 16 x 40 x 40: 49 against 46 us); inside the networks,
    // between other layers, taking them too is what measured faster (same box, two runs each: a detection network 1.752
    // -> 1.738 ms, another 0.820 -> 0.805 ms, a depthwise / pointwise network 0.772 -> 0.761 ms), and the networks decide.
    if (DT == EXHIP_F16 && g_exhip_options.pw_tile != 2) take = true;
    if (DT == EXHIP_F16 && ((g.c_bytes <= 128 && g.pixels <= 524288) || (g.c_bytes <= 256 && g.k <= 64 && g.pixels <= 131072))) take = true;
    if (g_exhip_options.pw != 2 && !take) return EXHIP_ERR_UNSUPPORTED;
    if (g.pixels <= 0 || g.c_bytes <= 0 || g.c_bytes % 32 != 0 || (g.slab_blocks != 2 && g.slab_blocks != 4) || g.k_stride % 8 != 0 || !pw_row_fits(4ll * g.k_stride))
        return EXHIP_ERR_UNSUPPORTED;
    // lane offsets are 32-bit: the input tensor and the packed weights must stay below the out-of-range sentinel
    const long long x_bytes = g.pixels * g.c_bytes;
    const long long n_ksteps = g.c_bytes / 32;
    const long long w_bytes = (long long)g.slabs * n_ksteps * g.slab_blocks * 1024;
    if (x_bytes >= kOutOfRange || w_bytes >= kOutOfRange || g.pixels * 4 * g.k_stride >= (1ll << 40)) return EXHIP_ERR_UNSUPPORTED;
    if (g.post_op && g.post_op != EXHIP_POST_PRELU && (g.post_op < 1 || g.post_op > 1 + EXHIP_UNARY_CLIP || g.post_op == 1 + EXHIP_UNARY_SIGMOID))
        return EXHIP_ERR_UNSUPPORTED;
    p.post_slope = g.post_slope;
    p.pixels = (unsigned)g.pixels; p.x_bytes = (unsigned)x_bytes; p.w_bytes = (unsigned)w_bytes;
    p.xs_b = g.c_bytes; p.n_ksteps = (int)n_ksteps; p.mts = g.slab_blocks;
    p.K = g.k; p.kstride = g.k_stride;
    p.act = g.act; p.post_relu = g.post_relu; p.post_op = g.post_op; p.post_slope_shared = g.post_slope_shared;
    p.residual_last = g.residual_last && has_residual;
    p.post_alpha = g.post_alpha; p.post_beta = g.post_beta;
    // every packed block that holds a channel below max(k, k_stride): pad channels of the output are written as zeros
    // (exact_k: only the blocks of the k channels themselves)
    const int kblocks = std::min(g.slabs * g.slab_blocks, (out_channels + 31) / 32);
    if constexpr (DT == EXHIP_F16)
        if (dw) return run_depthwise(ctx, *dw, p, kblocks, split_wins(DT, g, kblocks, (int)n_ksteps, false, 1));
    // 32 pixels x 64 channels a wave, 64 x 64 only where the option asks for it and no SIMD is left without a wave; a lone 32-channel
    // block takes 64 pixels
    if (split_wins(DT, g, kblocks, (int)n_ksteps, false, 1)) return launch_split<DT, false>(ctx, p, kblocks);
    if (kblocks == 1) return launch<DT, 1, 2>(ctx, p, kblocks);
    const long long waves64 = ((g.pixels + 63) / 64) * ((kblocks + 1) / 2);
    if (waves64 < 2048 || small_tile<DT>()) return launch<DT, 2, 1>(ctx, p, kblocks);
    return launch<DT, 2, 2>(ctx, p, kblocks);
}

}  // namespace

int exhip_conv1x1_f16_pw(exhip_ctx* ctx, const exhip_pw_geom& g, const uint16_t* x, const void* wp, const float* bias,
                         const uint16_t* residual, uint16_t* y, const exhip_pw_taps* taps, const exhip_pw_depthwise* dw) {
    PwParams p = {};
    p.x = reinterpret_cast<const char*>(x); p.wp = reinterpret_cast<const char*>(wp); p.bias = bias; p.residual = residual; p.y = y;
    return run_pw<EXHIP_F16>(ctx, g, p, 2, residual != nullptr, taps, dw);
}

int exhip_conv1x1_i8_pw(exhip_ctx* ctx, const exhip_pw_geom& g, const int8_t* x, const void* wp, const float* scale, const float* bias,
                        const float* residual, int8_t* y_i8, float* y_f32, const exhip_pw_taps* taps) {
    if (!scale || (!y_i8 && !y_f32) || g.k_stride % 16 != 0) return EXHIP_ERR_UNSUPPORTED;
    PwParams p = {};
    p.x = reinterpret_cast<const char*>(x); p.wp = reinterpret_cast<const char*>(wp); p.bias = bias; p.scale = scale;
    p.residual_f = residual; p.y_f = y_f32; p.y_q = y_i8; p.fs_out = g.fs_out;
    return run_pw<EXHIP_I8>(ctx, g, p, 1, residual != nullptr, taps);
}

int exhip_conv_f16_stem(exhip_ctx* ctx, const exhip_pw_geom& g, const exhip_pw_taps& t, int channels, const uint16_t* x, const float* mean, const float* factor,
                        const void* wp, const float* bias, uint16_t* y) {
    PwParams p = {};
    p.x = reinterpret_cast<const char*>(x); p.wp = reinterpret_cast<const char*>(wp); p.bias = bias; p.y = y;
    p.mean = mean; p.factor = factor;
    return run_stem<EXHIP_F16>(ctx, g, t, channels, p);
}

int exhip_conv_i8_stem(exhip_ctx* ctx, const exhip_pw_geom& g, const exhip_pw_taps& t, int channels, const float* x, const float* mean, const float* factor,
                       float fs_in, const void* wp, const float* scale, const float* bias, int8_t* y_i8, float* y_f32) {
    PwParams p = {};
    p.x = reinterpret_cast<const char*>(x); p.wp = reinterpret_cast<const char*>(wp); p.scale = scale; p.bias = bias; p.y_q = y_i8; p.y_f = y_f32;
    p.mean = mean; p.factor = factor; p.fs_in = fs_in; p.fs_out = g.fs_out;
    return run_stem<EXHIP_I8>(ctx, g, t, channels, p);
}

int exhip_pw_runs_f16(const exhip_pw_geom& g, int start[5]) {
    const int n_ksteps = g.c_bytes / 32, kblocks = std::min(g.slabs * g.slab_blocks, (std::max(g.k, g.k_stride) + 31) / 32);
    if (!split_wins(EXHIP_F16, g, kblocks, n_ksteps, false, 1)) return 1;
    for (int i = 0; i <= kSplit; ++i) start[i] = split_start(n_ksteps, n_ksteps % 2 == 0, i);
    return kSplit;
}

bool exhip_pw_splits_f16(long long pixels, int c_bytes, int k, int k_stride, int n_ksteps, int stride) {
    exhip_pw_geom g = {};
    g.pixels = pixels; g.c_bytes = c_bytes;
    return g_exhip_options.pw != 0 && g_exhip_options.direct != 0 && split_wins(EXHIP_F16, g, (std::max(k, k_stride) + 31) / 32, n_ksteps, true, stride);
}

int exhip_pw_pair(exhip_ctx* ctx, int (*layer)(exhip_ctx*, const void*), const void* first, const void* second) {
    return exhip_run_pair(ctx, &t_collect, layer, first, second, [ctx](const exhip_waiting<PwParams>* w) {
        if (w[0].dt != w[1].dt) return EXHIP_ERR_UNSUPPORTED;
        PwTwo q;
        for (int i = 0; i < 2; ++i) q.p[i] = w[i].p, q.kind[i] = w[i].kind, q.groups[i] = w[i].groups;
        const dim3 grid(w[0].groups + w[1].groups);
        if (w[0].dt == EXHIP_I8) hipLaunchKernelGGL(conv_pw_two_kernel<EXHIP_I8>, grid, dim3(256), 0, ctx->stream, q);
        else hipLaunchKernelGGL(conv_pw_two_kernel<EXHIP_F16>, grid, dim3(256), 0, ctx->stream, q);
        EXHIP_LAUNCH_CHECK();
        return 0;
    });
}
