// conv3x3_staged_kernel: layers with a 3x3 filter on NHWC tensors, fp16 at stride 1 and 2, int8 at stride 1, the input under a run of output pixels staged in LDS.
//
// The tapped form of conv_pw.hip reads every pixel up to nine times through a CU's address path, a KiB and a half for each MFMA: 96 cycles of L1 for 32 of the matrix unit.
// The lean kernel (conv_i8_lean.hip) stages patches of up to 256 pixels x 64 channels, one a CU: a launch of 300 patches is two rounds, maps that patches do not divide
// waste lanes, and four waves that all wait for the same barrier hide nothing from each other. Here a group's 64 to 256 pixels are neighbours
// in a list of the output's vertical strips, row by row, whatever map they belong to (strips.h), three groups share a CU, and
// up to four waves share a run's sums where the launch is small. Pixels come from LDS (64 x 64 a wave: half a KiB for each MFMA, as
// much of the weights from the caches, a filter row's six k-steps ahead); a run's input is staged 64 to 256 bytes a pixel at a time, the
// next piece on its way into registers meanwhile. At stride 2 a staged row holds its even columns first, so that neighbouring lanes read neighbouring pixels.
// What bounds it: fp16 the matrix units, 56 cycles an MFMA with random data at 16 x 40 x 40 128 -> 128 (their power allows about 48), of 12 us 8, the rest
// the chain from launch to the first products, 5000 cycles, and from the last ones to the stores, 2000 to 3700; int8, with half the MFMAs,
// those two. us, the other kernels -> this one: the rule below.
// Three waves a SIMD leave 168 registers: 72 of the 75 instantiations keep 2 to 7 of theirs in scratch, 12 to 32 bytes a lane.
//
// Sums of a group whose waves share them run in another order than the general kernel's, the same every time.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <mutex>

#include "conv_pw_epilogue.h"
#include "conv_staged.h"
#include "strips.h"

namespace {

constexpr int kLdsLimit = 160 * 1024;

struct StagedParams {
    PwParams f;
    exhip_divisor by_groups;
    exhip_strip_list list;
    int subs, chunks;              // pieces of 64 bytes of a pixel, and what is staged of them at a time
    int tap_w, half_w;             // bytes of the weights from a tap to the next one, and from a piece's first half to its second
    int table_b;                   // bytes of the table in front of the staged pixels
};

// Rows of 32 pixels anywhere in the output from an LDS tile to memory: CHUNKS 16-byte pieces a row, neighbouring lanes on neighbouring pieces.
template <int CHUNKS>
__device__ __forceinline__ void store_scattered(const char* tile, int pitch, __amdgpu_buffer_rsrc_t y, unsigned pix, int row_bytes, int ch_bytes, int bytes, int lane) {
    const int row = lane / CHUNKS, col = (lane % CHUNKS) * 16;
#pragma unroll
    for (int j = 0; j < CHUNKS / 2; ++j) {
        const int r = j * (64 / CHUNKS) + row;
        const unsigned to = (unsigned)__builtin_amdgcn_ds_bpermute(r * 4, (int)pix);
        const v4i t = *reinterpret_cast<const v4i*>(tile + r * pitch + col);
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(__attribute__((ext_vector_type(4))) unsigned int, t), y,
                                               to != 0xffffffffu && col < bytes ? (int)(to * (unsigned)row_bytes) + ch_bytes + col : kOutOfRange, 0, 0);
    }
}

// A wave's sums to results, as pw_epilogue (conv_pw_epilogue.h), for pixels that are not neighbours in memory: pix[n] is the lane's of block n.
template <int DT, int MT, int NT, typename EP, typename ACC>
__device__ __forceinline__ void scattered_epilogue(const PwParams& p, const ACC (&acc)[MT][NT], const unsigned (&pix)[NT], int kb0, int lane, char* lds) {
    constexpr bool I8 = DT == EXHIP_I8, ANY = EP::any;
    constexpr int ES = I8 ? 4 : 2;
    const int half = lane >> 5, row = lane & 31;
    char* const tile = lds + param_bytes(MT);
    const int k_end = pw_channel_end(p.K, p.kstride, 0);
    const bool shortcut = ANY ? (I8 ? p.residual_f != nullptr : p.residual != nullptr) : EP::res != 0;
    auto view = [&](const void* base, int es) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, base ? (int)(p.pixels * (unsigned)p.kstride) * es : 0, kRsrcWord3); };
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        const bool mine = pix[n] != 0xffffffffu;
        auto place = [&](int ch, int es) { return mine && ch < k_end ? (int)(pix[n] * (unsigned)p.kstride + ch) * es : kOutOfRange; };
        v4i r[MT][ES];
        if (shortcut) {
            const __amdgpu_buffer_rsrc_t rr = view(I8 ? (const void*)p.residual_f : (const void*)p.residual, ES);
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int q = 0; q < ES; ++q)
                    r[m][q] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rr, place((kb0 + m) * 32 + half * 16 + q * (16 / ES), ES), 0, 0));
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
                const int word = r[m][I8 ? e >> 2 : e >> 3][I8 ? e & 3 : (e >> 1) & 3];
                if constexpr (I8) return __builtin_bit_cast(float, word);
                else return exhip_h2f((uint16_t)(((uint32_t)word >> ((e & 1) * 16)) & 0xffff));
            });
            if (kb * 32 + 32 > p.K) {  // pad channels hold zeros
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    if (ch0 + e >= p.K) v[e] = 0.f;
            }
            if constexpr (I8) {
                if (p.y_f) {
                    constexpr int pitch = 128 + 16;
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const v4f o = {v[q * 4], v[q * 4 + 1], v[q * 4 + 2], v[q * 4 + 3]};
                        *reinterpret_cast<v4f*>(tile + row * pitch + half * 64 + q * 16) = o;
                    }
                    store_scattered<8>(tile, pitch, view(p.y_f, 4), pix[n], p.kstride * 4, kb * 128, (k_end - kb * 32) * 4, lane);
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
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(__attribute__((ext_vector_type(4))) unsigned int, o), view(p.y_q, 1), place(ch0, 1), 0, 0);
                }
            } else {
                constexpr int pitch = MT * 64 + 16;
                v4i o[2];
#pragma unroll
                for (int e = 0; e < 8; ++e) o[e >> 2][e & 3] = (int)exhip_round_pair(v[2 * e], v[2 * e + 1]);
                *reinterpret_cast<v4i*>(tile + row * pitch + m * 64 + half * 32) = o[0];
                *reinterpret_cast<v4i*>(tile + row * pitch + m * 64 + half * 32 + 16) = o[1];
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (!I8)
            store_scattered<MT * 4>(tile, MT * 64 + 16, view(p.y, 2), pix[n], p.kstride * 2, kb0 * 64, (k_end - kb0 * 32) * 2, lane);
    }
}

// A wave's tile is 32 * MT channels x 32 * NT pixels; WP waves side by side make a group's run of pixels, WK share its sums. S: the stride; SUBS pieces of 64
// bytes of a pixel are staged at a time.
template <int DT, int MT, int NT, int WK, int WP, int S, int SUBS, typename EP>
__global__ __launch_bounds__(64 * WK * WP, 3) void conv3x3_staged_kernel(const StagedParams q) {
    exhip_touch_args(q);
    const PwParams& p = q.f;
    constexpr int WAVES = WK * WP, THREADS = 64 * WAVES, RUN = 32 * NT * WP;
    constexpr int BYTES = SUBS * 64, PIECES = BYTES / 16, PASS = THREADS / PIECES, PITCH = BYTES + 16;  // of a staged pixel
    constexpr int BATCH = 6;    // passes whose pixels are on the way at a time
    constexpr int ROW = 6;      // k-steps of a filter row in a piece
    extern __shared__ __attribute__((aligned(16))) char lds_all[];
    int* const table = reinterpret_cast<int*>(lds_all);   // where the staged pixels lie in the input
    char* const stage = lds_all + q.table_b;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), half = lane >> 5;
    const int part = wave % WK, side = wave / WK;
    unsigned bid = blockIdx.x;
    {
        const unsigned per = gridDim.x >> 3;  // one contiguous run of items per XCD
        if (bid < (per << 3)) bid = (bid & 7) * per + (bid >> 3);
    }
    const unsigned tile = __builtin_amdgcn_readfirstlane(q.by_groups(bid));
    const int kb0 = __builtin_amdgcn_readfirstlane((int)(bid - tile * p.ch_groups) * MT);
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(p.x), 0, (int)p.x_bytes, kRsrcWord3);
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(p.wp), 0, (int)p.w_bytes, kRsrcWord3);

    // weights: a unit is a filter row's taps of a piece, two k-steps each (conv_igemm.hip's packing, in chunks of a piece or of half a piece)
    const int w_step = p.mts * 1024, slab = kb0 >> (p.mts >> 1);
    const int w_base = (slab * p.n_ksteps * p.mts + (kb0 & (p.mts - 1))) * 1024;
    v4i a[ROW][MT];
    auto request = [&](int i, int unit) {  // unit < 0: nothing
        const int voff = unit < 0 ? kOutOfRange : lane * 16;
#pragma unroll
        for (int m = 0; m < MT; ++m) a[i][m] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(wr, voff + m * 1024, unit < 0 ? 0 : unit + (i >> 1) * q.tap_w + (i & 1) * q.half_w, 0));
    };
    auto unit_at = [&](int unit) { return w_base + unit / 3 * (18 * w_step) + unit % 3 * 3 * q.tap_w; };
    auto units_of = [&](int chunk) { return (chunk * SUBS + SUBS <= q.subs ? SUBS : q.subs - chunk * SUBS) * 3; };
    auto first_unit = [&](int chunk) { return units_of(chunk) * part / WK; };

    // the staged rows: those under the run's first pixel to those under its last
    const unsigned run0 = tile * RUN;
    const int first_row = __builtin_amdgcn_readfirstlane(q.list.template where<S>(run0, p.out_h, p.out_w).row);
    const int last_row = __builtin_amdgcn_readfirstlane(q.list.template where<S>(run0 + RUN - 1, p.out_h, p.out_w).row) + 2;
    const int staged = (last_row - first_row + 1) * q.list.staged_cols;
    const int even_cols = (q.list.staged_cols + 1) >> 1;  // S == 2: a row's even columns come first
    for (int i = threadIdx.x; i < staged; i += THREADS) table[i] = (int)q.list.template staged_pixel<S>(i, first_row, p.in_h, p.in_w, p.pad_t, p.pad_l, p.xs_b, kOutOfRange);
    __syncthreads();
    v4i x[BATCH];
    const int my_piece = threadIdx.x % PIECES, my_pixel = threadIdx.x / PIECES;
    auto load_batch = [&](int first, int chunk) {
#pragma unroll
        for (int i = 0; i < BATCH; ++i) {
            const int at = first + i * PASS + my_pixel;
            x[i] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(xr, at < staged && chunk * BYTES + my_piece * 16 < p.xs_b ? table[at] + my_piece * 16 : kOutOfRange, chunk * BYTES, 0));
        }
    };
    auto store_batch = [&](int first) {
#pragma unroll
        for (int i = 0; i < BATCH; ++i) {
            const int at = first + i * PASS + my_pixel;
            if (at < staged) *reinterpret_cast<v4i*>(stage + at * PITCH + my_piece * 16) = x[i];
        }
    };
    load_batch(0, 0);
#pragma unroll
    for (int i = 0; i < ROW; ++i) request(i, unit_at(first_unit(0)));
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
    }
    // the wave's pixels: their place in the staged rows, and in the output
    const char* b_at[NT];
    unsigned pix[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        const auto w = q.list.template where<S>(run0 + (side * NT + n) * 32 + (lane & 31), p.out_h, p.out_w);
        pix[n] = w.pix;
        b_at[n] = stage + ((w.row - first_row) * q.list.staged_cols + w.x) * PITCH + half * 16;
    }
    const int tap_row = q.list.staged_cols * PITCH, tap_col[3] = {0, S == 2 ? even_cols * PITCH : PITCH, S == 2 ? PITCH : 2 * PITCH};
    typedef typename std::conditional<DT == EXHIP_I8, v16i, v16f>::type acc_t;
    typedef typename std::conditional<DT == EXHIP_I8, v4i, v4f>::type four_t;
    acc_t acc[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[m][n][e] = 0;
    for (int first = 0;;) {
        store_batch(first);
        first += BATCH * PASS;
        if (first >= staged) break;
        load_batch(first, 0);
    }
    __syncthreads();

    v4i b[3][NT];
    auto fetch = [&](v4i (&to)[NT], int at) {
#pragma unroll
        for (int n = 0; n < NT; ++n) to[n] = *reinterpret_cast<const v4i*>(b_at[n] + at);
    };
#pragma unroll 1
    for (int chunk = 0; chunk < q.chunks; ++chunk) {
        const bool more = chunk + 1 < q.chunks;
        if (more) load_batch(0, chunk + 1);
        const int units = units_of(chunk), u1 = units * (part + 1) / WK, base = chunk * SUBS * 3;
        int u = units * part / WK, r = u % 3, row_at = u / 3 * 64 + r * tap_row;
        const int then = more ? unit_at(base + SUBS * 3 + first_unit(chunk + 1)) : -1;
        if (u < u1) fetch(b[0], row_at);
#pragma unroll 1
        for (; u < u1; ++u) {
            const int next = u + 1 < u1 ? unit_at(base + u + 1) : then;
            int row_next = row_at;
            if (u + 1 < u1) {
                row_next = ++r == 3 ? row_at + 64 - 2 * tap_row : row_at + tap_row;
                if (r == 3) r = 0;
            }
#pragma unroll
            for (int i = 0; i < ROW; ++i) {
                fetch(b[(i + 1) % 3], i + 1 == ROW ? row_next : row_at + tap_col[(i + 1) / 2 % 3] + (i + 1) % 2 * 32);
                __builtin_amdgcn_sched_barrier(0);  // (the reads would sink to where they are used)
#pragma unroll
                for (int m = 0; m < MT; ++m)
#pragma unroll
                    for (int n = 0; n < NT; ++n) {
                        if constexpr (DT == EXHIP_I8) acc[m][n] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[i][m], b[i % 3][n], acc[m][n], 0, 0, 0);
                        else acc[m][n] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, a[i][m]), __builtin_bit_cast(v8h, b[i % 3][n]), acc[m][n], 0, 0, 0);
                    }
                request(i, next);
                __builtin_amdgcn_sched_barrier(0);
            }
            row_at = row_next;
        }
        if (more) {
            __syncthreads();
            for (int first = 0;;) {
                store_batch(first);
                first += BATCH * PASS;
                if (first >= staged) break;
                load_batch(first, chunk + 1);
            }
        }
        __syncthreads();
    }

    // the staged pixels are no longer read
    constexpr int OM = WK <= NT ? MT : MT * NT / WK, ON = WK <= NT ? NT / WK : 1, SPLIT = MT / OM;  // the blocks a wave finishes; waves to an NT
    const int own_n = WK <= NT ? part * ON : part / SPLIT, own_m = WK <= NT ? 0 : part % SPLIT * OM;
    // a wave's inbox: the others' sums of the blocks it finishes; later what it keeps to itself
    constexpr int BOX = (WK - 1) * OM * ON * 4096 > wave_bytes(DT, OM) ? (WK - 1) * OM * ON * 4096 : wave_bytes(DT, OM);
    char* const mine = lds_all + wave * BOX;
    acc_t own[OM][ON];
    unsigned own_pix[ON];
    if constexpr (WK == 1) {
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            own_pix[n] = pix[n];
#pragma unroll
            for (int m = 0; m < MT; ++m) own[m][n] = acc[m][n];
        }
    } else {
        // the waves' sums meet in LDS and are added in their order
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const int to = WK <= NT ? n / ON : n * SPLIT + m / OM, block = WK <= NT ? n % ON * MT + m : m % OM;  // whose it is, and which of its
                if (to == part) continue;
                char* const box = lds_all + (side * WK + to) * BOX + ((part - (part > to)) * (OM * ON) + block) * 4096;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const acc_t& c = acc[m][n];
                    *reinterpret_cast<four_t*>(box + v * 1024 + lane * 16) = four_t{c[v * 4], c[v * 4 + 1], c[v * 4 + 2], c[v * 4 + 3]};
                }
            }
        __syncthreads();
#pragma unroll
        for (int n = 0; n < ON; ++n) {
            own_pix[n] = 0;
#pragma unroll
            for (int i = 0; i < NT; ++i) own_pix[n] = own_n + n == i ? pix[i] : own_pix[n];
#pragma unroll
            for (int m = 0; m < OM; ++m) {
                acc_t here = acc[m][n];
#pragma unroll
                for (int i = 0; i < NT; ++i)
#pragma unroll
                    for (int j = 0; j < MT; ++j)
                        if (own_n + n == i && own_m + m == j) here = acc[j][i];
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    four_t sum = {};
#pragma unroll
                    for (int w = 0; w < WK; ++w) {
                        four_t t = {here[v * 4], here[v * 4 + 1], here[v * 4 + 2], here[v * 4 + 3]};
                        if (w != part) t = *reinterpret_cast<const four_t*>(mine + ((w - (w > part)) * (OM * ON) + n * OM + m) * 4096 + v * 1024 + lane * 16);
                        sum = w == 0 ? t : sum + t;
                    }
#pragma unroll
                    for (int e = 0; e < 4; ++e) own[m][n][v * 4 + e] = sum[e];
                }
            }
        }
    }
    const int at = lane - own_m * 32;
    if (at >= 0 && at < OM * 32 && lane < MT * 32) {
#pragma unroll
        for (int i = 0; i < kParams; ++i) *reinterpret_cast<float*>(mine + (i * OM * 32 + at) * 4) = par[i];
    }
    if (kb0 + own_m > 0 && !pw_block_exists(kb0 + own_m, pw_channel_end(p.K, p.kstride, 0))) return;
    scattered_epilogue<DT, OM, ON, EP>(p, own, own_pix, kb0 + own_m, lane, mine);
}

std::mutex g_attr_mutex;

// Staged pixels with which three groups share a CU, as many as their registers allow.
int most_staged(int pitch) { return (kLdsLimit / 3 - 1280 - 16) / (pitch + 4); }

struct Launch {
    unsigned groups;
    int threads, lds;
};

template <void (*KERNEL)(const StagedParams)>
int launch(exhip_ctx* ctx, const StagedParams& q, const Launch& l) {
    {
        static unsigned long long attr_set = 0;
        std::lock_guard<std::mutex> lock(g_attr_mutex);
        const unsigned long long bit = 1ull << (ctx->device & 63);
        if (!(attr_set & bit)) {
            EXHIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(KERNEL), hipFuncAttributeMaxDynamicSharedMemorySize, kLdsLimit));
            attr_set |= bit;
        }
    }
    hipLaunchKernelGGL(KERNEL, dim3(l.groups), dim3(l.threads), l.lds, ctx->stream, q);
    EXHIP_LAUNCH_CHECK();
    return 0;
}

constexpr int kMt = 2, kNt = 2, kForms = 3;
struct Form {
    int wk, wp, subs;  // waves that share a run's sums and side by side, pieces staged at a time
    constexpr int run() const { return 32 * kNt * wp; }
    constexpr int pitch() const { return subs * 64 + 16; }
    constexpr int own_m() const { return wk <= kNt ? kMt : kMt * kNt / wk; }
    constexpr int own() const { return kMt * kNt / wk; }  // blocks a wave finishes
    int lds(int dt, int staged) const {
        return std::max((staged * 4 + 15) / 16 * 16 + staged * pitch(), wk * wp * std::max((wk - 1) * own() * 4096, wave_bytes(dt, own_m())));
    }
};
constexpr Form kForm[2][kForms] = {{{1, 4, 1}, {2, 2, 2}, {4, 1, 4}}, {{1, 4, 1}, {2, 2, 1}, {4, 1, 2}}};  // at stride 1 and 2

struct Plan {
    int form = -1;
    exhip_strips strips;
    double time = 0;  // us
};

// A model of the launch, fitted per type to 171 layers (1 to 64 maps of 7 x 7 to 320 x 320, 64 to 512 channels) under six to nine kinds of layers behind, 4.5 %
// off on average; the form it picks is 0.5 % slower than the fastest on average.
constexpr double kModel[2][13] = {
    // a group's start, a stage's and its per batch, an MFMA, meeting sums, a block's results and what lies behind them: a wave's chain; busy per MFMA, block, what
    // lies behind, stage; how much a wave beside it costs; the launch
    {2.41, 0.59, 0.59, 0.0128, 0.03, 0.03, 0.37, 0.0169, 0.11, 0.41, 0.56, 0.26, 2.65},    // int8
    {2.23, 0.53, 0.59, 0.0154, 0.22, 0.0, 0.08, 0.0181, 0.24, 0.10, 0.63, 0.10, 2.79}};    // fp16

Plan choose(int dt, const PwParams& p, long long images, int subs, int kblocks) {
    const double* const t = kModel[dt == EXHIP_F16];
    const bool shortcut = p.residual || p.residual_f;
    const double behind = (p.post_op ? 1.0 : p.act || p.post_relu ? 0.3 : 0.1) + (shortcut ? 0.7 : 0) + (dt == EXHIP_I8 && p.y_f ? 0.9 : 0);
    const double out_bytes = dt == EXHIP_F16 ? (shortcut ? 4 : 2) : (p.y_q ? 1 : 0) + (p.y_f ? 4 : 0) + (shortcut ? 4 : 0);
    const double bytes = (double)p.pixels * p.kstride * out_bytes + p.x_bytes;
    Plan best;
    for (int i = 0; i < kForms; ++i) {
        const Form& f = kForm[p.stride - 1][i];
        const exhip_strips s = exhip_choose_strips(p.out_h, p.out_w, p.stride, images, f.run(), most_staged(f.pitch()), 0);
        const int lds = (f.lds(dt, s.staged) + 1279) / 1280 * 1280;
        if (lds > kLdsLimit) continue;
        const long long groups = s.tiles * ((kblocks + 1) / 2), slots = 256ll * std::min(kLdsLimit / lds, 3), full = groups / slots;
        const double steps = subs * 18.0 / f.wk * 4, chunks = (subs + f.subs - 1) / f.subs, batches = s.staged * f.subs * 4 / 1536.0;
        const double chain = t[0] + chunks * (t[1] + t[2] * batches) + steps * t[3] + (f.wk > 1 ? t[4] : 0) + f.own() * (t[5] + t[6] * behind);
        const double busy = steps * t[7] + f.own() * (t[8] + t[9] * behind) + chunks * batches * t[10];
        auto round = [&](long long n) {
            const double w = (double)((n + 255) / 256);
            return n ? std::max(chain * (1 + t[11] * (w - 1)), busy * w + t[0]) : 0.;
        };
        const double time = t[12] + std::max(full * round(slots) + round(groups - full * slots), bytes / 5.5e6);
        if (best.form < 0 || time < best.time) {
            best.form = i;
            best.strips = s;
            best.time = time;
        }
    }
    return best;
}

template <int DT, int S, int WK, int WP, int SUBS>
int go(exhip_ctx* ctx, StagedParams& q, long long images, int kblocks, const exhip_strips& s) {
    constexpr int MT = kMt, NT = kNt, WAVES = WK * WP;
    PwParams& p = q.f;
    q.chunks = (q.subs + SUBS - 1) / SUBS;
    q.table_b = (s.staged * 4 + 15) / 16 * 16;
    const int lds = Form{WK, WP, SUBS}.lds(DT, s.staged);
    if (lds > kLdsLimit) return EXHIP_ERR_UNSUPPORTED;
    q.list.set(s, p.out_h, S, images);
    p.ch_groups = (unsigned)((kblocks + MT - 1) / MT);
    q.by_groups.set(p.ch_groups);
    const long long items = s.tiles * p.ch_groups;
    if (items >= (1ll << 31) - 4) return EXHIP_ERR_UNSUPPORTED;
    const Launch l = {(unsigned)items, 64 * WAVES, lds};
    const bool shortcut = DT == EXHIP_I8 ? p.residual_f != nullptr : p.residual != nullptr;
    const int res = !shortcut ? 0 : p.residual_last ? 2 : 1;
    int act = p.act, post = p.post_relu ? kPostRelu : kPostNone;
    if (DT == EXHIP_I8 && act == 1 && !res && !p.post_op) act = 0, post = kPostRelu;  // (nothing is rounded between the two)
    if (p.post_op) post = post == kPostNone && p.post_op == 1 + EXHIP_UNARY_HARDSWISH ? kPostHardSwish : post == kPostNone && p.post_op == EXHIP_POST_PRELU ? kPostPrelu : -1;
#define STAGED_AS(POST, RES) \
    if (act == 0 && post == POST && res == RES) return launch<conv3x3_staged_kernel<DT, MT, NT, WK, WP, S, SUBS, Ep<0, POST, RES>>>(ctx, q, l);
    STAGED_AS(kPostNone, 0)
    STAGED_AS(kPostHardSwish, 0)
    STAGED_AS(kPostRelu, 0)
    STAGED_AS(kPostHardSwish, 2)
    STAGED_AS(kPostRelu, 1)
    if constexpr (DT == EXHIP_F16) {
        STAGED_AS(kPostPrelu, 0)
        if (act == 1 && post == kPostNone && res == 0) return launch<conv3x3_staged_kernel<DT, MT, NT, WK, WP, S, SUBS, Ep<1, kPostNone, 0>>>(ctx, q, l);
        STAGED_AS(kPostNone, 1)
    } else {
        STAGED_AS(kPostRelu, 2)
    }
#undef STAGED_AS
    return launch<conv3x3_staged_kernel<DT, MT, NT, WK, WP, S, SUBS, EpAny>>(ctx, q, l);
}

template <int DT, int S, int FORM>
int go_form(exhip_ctx* ctx, StagedParams& q, long long images, int kblocks, const exhip_strips& s) {
    constexpr Form f = kForm[S - 1][FORM];
    return go<DT, S, f.wk, f.wp, f.subs>(ctx, q, images, kblocks, s);
}

template <int DT, int S>
int pick(exhip_ctx* ctx, StagedParams& q, long long images, int kblocks, const Plan& plan) {
    if (plan.form == 0) return go_form<DT, S, 0>(ctx, q, images, kblocks, plan.strips);
    if (plan.form == 1) return go_form<DT, S, 1>(ctx, q, images, kblocks, plan.strips);
    return go_form<DT, S, 2>(ctx, q, images, kblocks, plan.strips);
}

// A thread keeps the plans of its last layers: the search takes a few microseconds.
Plan plan_of(int dt, const PwParams& p, long long images, int subs, int kblocks) {
    const int key[] = {dt, (int)images, p.out_h, p.out_w, p.stride, subs, kblocks, p.post_op, p.act, p.post_relu, (p.y_f ? 1 : 0) + (p.y_q ? 2 : 0) + (p.residual || p.residual_f ? 4 : 0)};
    constexpr int kKey = sizeof(key) / sizeof(key[0]);
    struct Entry {
        int key[kKey];
        Plan plan;
    };
    static thread_local Entry cache[64] = {};
    unsigned at = 0;
    for (int k : key) at = at * 31 + (unsigned)k;
    Entry& e = cache[(at ^ at >> 8) % 64];
    if (e.plan.form < 0 || !std::equal(key, key + kKey, e.key)) {
        e.plan = choose(dt, p, images, subs, kblocks);
        std::copy(key, key + kKey, e.key);
    }
    return e.plan;
}

}  // namespace

// Whether this kernel is the faster one for a layer. Ratios are the time of the kernel that would run it otherwise to this one's, over 171 layers; `work` counts blocks of 32 pixels x 32
// channels times k-steps.
//  * Few blocks: the split form (conv_pw.hip), whose tiles of 32 pixels share a CU by twos and fours (fp16 72 k-steps 502 blocks 0.78, 588 1.06; 36 k-steps 926
//    blocks 0.85, 1263 1.22).
//  * An odd number of pieces at stride 1 leaves the last stage of the forms for small launches, two or four pieces, partly empty. Below 126 k-steps (from there on the split form's own
//    waves are the longer ones: seven pieces 1.05 to 1.2) such layers stay with the split form up to 704 of its groups of two blocks, in either type: three pieces fp16 160 -> 320 at
//    10 x 13 x 13 8.0 there and 9.1 here, 96 -> 128 at 50 x 14 x 14 8.9 and 9.3, 96 -> 96 at 18 x 25 x 25, 704 groups, equal; five int8 320 -> 128 at 1 x 93 x 93 11.2 and 11.8, at
//    49 x 13 x 13 11.0 and 12.3. (Two and four pieces 0.95 to 1.2 between 512 and 704.) One piece is all staging: up to two rounds of 512 groups (fp16 32 -> 160 at
//    50 x 12 x 11 4.8 there and 6.6 here, 32 -> 352 at 2 x 52 x 52 5.8 and 7.5; equal from there on).
//  * fp16 at stride 1: everything else that the lean kernel cannot take, 1.04 to 1.6; what it can where its rounds of 256 patches of 256 pixels x 64 channels
//    take longer: 128 -> 128 at 8 x 40 x 40 13.6 -> 10.4 us, 256 -> 256 at 16 x 20 x 20 20.7 -> 14.8, 64 -> 128 at 11 x 151 x 151 77 -> 47;
//    its full rounds are 1 to 8 % shorter (64 -> 64 at 64 x 56 x 56, 128 -> 128 at 8 x 80 x 80).
//  * fp16 at stride 2: from 72 k-steps and 1280 blocks on 1.0 to 1.8 (128 -> 256 at 4 x 80 x 80 15.5 -> 12.3, 256 -> 512 at 32 x 40 x 40 73 -> 52; 256 -> 256
//    at 64 x 14 x 14, 784 blocks, 0.97); fewer k-steps on few output channels (64 -> 64 at 9 x 146 x 146 1.24) and very many blocks (32 -> 64 at
//    16 x 320 x 320 51.7 -> 45.6, 64 -> 128 at 32 x 160 x 160 1.14, at 64 x 56 x 56, 6272, 0.82).
//  * int8 at stride 1, where four waves of the lean kernel spend most of their time behind the products: an activation layer, none, or a float32 result beside
//    the int8 one from 36 k-steps on 1.0 to 2.0 (128 -> 128 at 8 x 80 x 80 with HardSwish 24.8 -> 14.6, 256 -> 256 at 16 x 20 x 20 12.9 -> 9.7), 18 k-steps without
//    float32 results 1.02 to 1.6, with them from 80 K of work on (1.03 to 1.4, below 0.96 to 1.0). A shortcut with ReLU: 1.0 to 1.3 up to 128 K of work,
//    beyond only what the lean kernel cannot take (64 -> 64 0.8, 192 -> 64 at 7 x 92 x 92 0.85). A ReLU alone, which the lean kernel has forms for: from 72 k-steps on
//    1.06 to 1.19 up to 128 K, 0.74 to 0.98 beyond and below; ragged channels, which it cannot take, 0.98 to 1.17.
//    Below 126 k-steps the split form, whose waves share a tile's steps, as long as its groups of two blocks are one round of 512 (384 -> 368 at 4 x 26 x 26
//    10.6 there and 12.3 here, 192 -> 352 at 12 x 14 x 14 6.5 and 7.4, 320 -> 128 at 3 x 41 x 41 8.8 and 9.2; even at 72 k-steps; from 126 on 1.03 to 1.2 here,
//    512 -> 64 at 12 x 30 x 30 12.0 and 10.1), 18 and 36 k-steps from 46 K of work on (64 -> 352 at 35 x 14 x 14, 42 K, 0.96).
//    Channels in odd thirty-twos, of which half a piece of products is for nothing and which the lean kernel has no form for: from 160 on 1.1 to 2.0
//    (160 -> 96 at 2 x 80 x 80 with HardSwish 16.5 -> 8.9, with a ReLU 12.3 -> 9.1; 760 blocks 0.94, 784 1.12), 96 where the launch is large (96 -> 160 at
//    8 x 66 x 66 18.0 -> 14.1, with a ReLU 0.95; 1800 blocks 0.9), 32 never (0.7 to 0.9).
//  * int8 at stride 2: 0.7 to 1.3 without a line between them; left alone.
bool exhip_staged_wins(int dt, const exhip_pw_geom& g, int stride, int n_ksteps, bool shortcut, bool y_f) {
    const exhip_options& o = g_exhip_options;  // (an option that pins another kernel's form is for that kernel)
    if (o.staged != 1) return o.staged > 1;
    if (o.direct != 1 || o.pw_split != 1 || o.pw_tile != 0 || o.lean != 4 || o.lean_f16 != 1 || o.lean_cfg != 0 || o.lean_wres != 1 || o.lean_groups != 0 || o.force_variant >= 0 ||
        o.force_chunk != 0 || o.force_rs != 0 || o.force_abufs != 0 || o.force_splits != 0)
        return false;
    const int kblocks = std::min(g.slabs * g.slab_blocks, (std::max(g.k, g.k_stride) + 31) / 32), ks = n_ksteps;
    const long long blocks = (g.pixels + 31) / 32 * kblocks, work = blocks * ks;
    if (blocks <= (dt == EXHIP_F16 && ks < 72 ? 1024 : kStagedBlocks)) return false;
    const bool ragged = g.c_bytes % 128 == 64 && ks < 126;  // an odd number of pieces: the last stage of two or four is not full
    const long long pairs = (g.pixels + 31) / 32 * ((kblocks + 1) / 2);
    if (ragged && stride == 1 && pairs <= (ks <= 18 ? 1024 : 704)) return false;
    if (dt == EXHIP_F16) return stride == 1 || (ks >= 72 ? blocks > 1280 : (kblocks <= 3 && blocks >= 1536) || blocks >= 12288);
    if (stride == 2 || work < (ks <= 36 ? 46 : 41) * 1024) return false;
    if (g.c_bytes % 64 != 0) return ks >= 45 ? blocks > 768 : ks >= 27 && blocks > 4096 && (g.post_op || shortcut || y_f || !(g.act || g.post_relu));
    if (ks < 126 && pairs <= 512) return false;
    const bool mid = work <= 128 * 1024 || g.k % 64 != 0;
    if (g.post_op) return ks >= 36 || (!shortcut && !y_f) || work >= 80 * 1024;
    if (shortcut) return ks >= 36 && mid;
    if (y_f) return ks >= 36 || work >= 80 * 1024;
    if (g.act || g.post_relu) return (ks >= 72 || g.k % 64 != 0) && mid;
    return true;
}

int exhip_conv3x3_staged(exhip_ctx* ctx, int dt, const void* pw_params, long long images, int kblocks, int lean_tiles) {
    const PwParams& p = *static_cast<const PwParams*>(pw_params);
    const int option = g_exhip_options.staged, subs = (p.xs_b + 63) / 64;
    const int widest = dt == EXHIP_F16 ? 2 : p.y_f || p.residual_f ? 4 : 1;  // bytes of an output (or shortcut) value
    if ((long long)p.pixels * p.kstride * widest >= kOutOfRange || p.kh != 3 || p.kw != 3 || (p.stride != 1 && (p.stride != 2 || dt != EXHIP_F16)) ||
        (p.xs_b % 64 != 0 && dt != EXHIP_I8) || p.pool || p.group || p.exact || kblocks < 2)
        return EXHIP_ERR_UNSUPPORTED;
    Plan plan;
    if (option > 1) {
        plan.form = std::min(option - 2, kForms - 1);
        const Form& f = kForm[p.stride - 1][plan.form];
        plan.strips = exhip_choose_strips(p.out_h, p.out_w, p.stride, images, f.run(), most_staged(f.pitch()), 0);
    } else {
        plan = plan_of(dt, p, images, subs, kblocks);
        if (plan.form < 0) return EXHIP_ERR_UNSUPPORTED;
        if (lean_tiles) {  // (its groups walk their patches one after another; up to two each the fuller half decides)
            const double rounds = lean_tiles <= 512 ? (lean_tiles + 255) / 256 : lean_tiles / 256.;
            if (plan.time >= 0.92 * (4 + rounds * (1.3 + 0.119 * p.n_ksteps))) return EXHIP_ERR_UNSUPPORTED;
        }
    }
    StagedParams q = {};
    q.f = p;
    // (int8 pixels that end with half a piece: the other half is staged as zeros, whatever weights its products read. Behind the last slab's the packing has as many zeros:
    // to leave those requests out took 1.2 to 3 %.)
    if (p.xs_b % 64) q.f.w_bytes += (unsigned)exhip_staged_pad(p.mts);
    q.subs = subs;
    q.tap_w = p.mts * (p.chunk_b == 64 ? 2048 : 1024);
    q.half_w = p.mts * (p.chunk_b == 64 ? 1024 : 9 * 1024);
    if (dt == EXHIP_I8) return pick<EXHIP_I8, 1>(ctx, q, images, kblocks, plan);
    return p.stride == 1 ? pick<EXHIP_F16, 1>(ctx, q, images, kblocks, plan) : pick<EXHIP_F16, 2>(ctx, q, images, kblocks, plan);
}
