// The inner step of the convolutions' weight packings (host code): the 16-byte vectors of a block of 64 lanes, one per lane and
// filter tap, each of a few neighbouring input channels. The channels' taps lie side by side in the OIHW weights.
#pragma once
#include <string.h>

#include <cstddef>

template <typename T, int TAPS>
inline void exhip_pack_full(const T* src, int taps_any, char* out, size_t tap_bytes) {
    constexpr int kPer = 16 / sizeof(T);
    const int taps = TAPS ? TAPS : taps_any;
    for (int t = 0; t < taps; ++t) {
        T v[kPer];
        for (int e = 0; e < kPer; ++e) v[e] = src[e * taps + t];
        memcpy(out + t * tap_bytes, v, 16);
    }
}

// One lane: n channels from src on, zeros behind them.
template <typename T>
inline void exhip_pack_lane(const T* src, int n, int taps, char* out, size_t tap_bytes) {
    constexpr int kPer = 16 / sizeof(T);
    if (n == kPer) {
        if (taps == 1) memcpy(out, src, 16);
        else if (taps == 9) exhip_pack_full<T, 9>(src, taps, out, tap_bytes);
        else exhip_pack_full<T, 0>(src, taps, out, tap_bytes);
        return;
    }
    for (int t = 0; t < taps; ++t) {
        T v[kPer] = {};
        for (int e = 0; e < n; ++e) v[e] = src[e * taps + t];
        memcpy(out + t * tap_bytes, v, 16);
    }
}

// The 64 lanes of a 32-channel block, tap t's KiB at out + t * tap_bytes; row_source(rr, half, &n) is where lane half * 32 + rr's n
// channels begin. Host time of a 512 -> 512 layer, of a loop that tests every element -> of this, ms: 1x1 float32 0.90 -> 0.30, fp16
// 0.53 -> 0.20, int8 0.46 -> 0.10; 3x3 float32 2.8 -> 1.6, fp16 1.8 -> 1.25, int8 1.3 -> 1.15. The KiBs are put together in a buffer,
// since taps lie powers of two apart in the packing and would drive each other out of the first-level cache, and a row's next step
// is requested ahead: the 32 rows lie too far apart for the core to see them as streams (3x3 float32 3.6 without, int8 3.3 at stride 2).
template <typename T, typename F>
inline void exhip_pack_block(F row_source, int taps, char* out, size_t tap_bytes) {
    constexpr int kBuffered = 32;
    const bool buffered = taps > 1 && taps <= kBuffered;
    char buffer[kBuffered * 1024];
    char* const to = buffered ? buffer : out;
    const size_t step = buffered ? 1024 : tap_bytes;
    for (int rr = 0; rr < 32; ++rr)
        for (int half = 0; half < 2; ++half) {
            int n = 0;
            const T* src = row_source(rr, half, &n);
            for (int o = 0; n && o < 16 * taps; o += 64) __builtin_prefetch(reinterpret_cast<const char*>(src) + 32 * taps + o);
            exhip_pack_lane(src, n, taps, to + (half * 32 + rr) * 16, step);
        }
    if (buffered)
        for (int t = 0; t < taps; ++t) memcpy(out + t * tap_bytes, buffer + t * 1024, 1024);
}
