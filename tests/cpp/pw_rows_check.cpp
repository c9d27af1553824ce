// Walks the pointwise kernels' epilogue over shapes with the arithmetic the kernels themselves use (pw_rows.h): every 16-byte
// access that a view lets through lies inside the tensor, and together the stores cover each row's channels once.
#include <cstdio>
#include <vector>

#include "../../excalibur_amd/csrc/pw_rows.h"

namespace {
long long checked = 0;

// What the hardware does with an offset: dropped (false) at or beyond the view's size, an unsigned word.
bool lands(int view, int offset) { return (unsigned)offset + 16u <= (unsigned)view; }

int fail(const char* what, int k, int k_stride, int pixels, int kb, int row, int offset, int view) {
    std::printf("%s: k %d stride %d pixels %d block %d row %d offset %d view %d\n", what, k, k_stride, pixels, kb, row, offset, view);
    return 1;
}

// mt blocks to a wave (1: the split form's waves, one block of a pair each); es bytes a value
int walk(int k, int k_stride, bool exact, int pixels, int mt, int es) {
    const int end = pw_channel_end(k, k_stride, exact), kblocks = (end + 31) / 32, row_bytes = k_stride * es;
    const long long tensor = (long long)pixels * row_bytes;
    std::vector<int> stored((size_t)pixels * (row_bytes / 16), 0);
    for (int first = 0; first < pixels; first += 32) {
        const int rows = pixels - first < 32 ? pixels - first : 32;
        for (int kb = 0; kb < (kblocks + 1) / 2 * 2; kb += mt) {  // the last pair may reach beyond the last block
            if (mt == 1 && !pw_block_exists(kb, end)) {
                // nobody comes here; if somebody did, an empty view would drop all it has
                const int view = pw_view_bytes(rows, row_bytes, kb * 32 * es);
                if (view < 0 || lands(view, kPwOutOfRange)) return fail("view of a missing block", k, k_stride, pixels, kb, 0, kPwOutOfRange, view);
                continue;
            }
            const int at0 = kb * 32 * es, view = pw_view_bytes(rows, row_bytes, at0);
            if (view < 0 || lands(view, kPwOutOfRange)) return fail("view", k, k_stride, pixels, kb, 0, kPwOutOfRange, view);
            const long long origin = (long long)first * row_bytes + at0;
            for (int row = 0; row < 32; ++row)
                for (int byte = 0; byte < mt * 32 * es; byte += 16) {
                    ++checked;
                    const int read = pw_lane_offset(row, row_bytes, byte, (k_stride - kb * 32) * es);
                    if (lands(view, read) && origin + read + 16 > tensor) return fail("load", k, k_stride, pixels, kb, row, read, view);
                    const int write = pw_lane_offset(row, row_bytes, byte, (end - kb * 32) * es);
                    if (!lands(view, write)) continue;
                    if (origin + write + 16 > tensor) return fail("store", k, k_stride, pixels, kb, row, write, view);
                    ++stored[(origin + write) / 16];
                }
        }
    }
    for (int p = 0; p < pixels; ++p)
        for (int j = 0; j < row_bytes / 16; ++j)
            if (stored[(size_t)p * (row_bytes / 16) + j] != (j * 16 < end * es ? 1 : 0)) return fail("coverage", k, k_stride, pixels, j, p, 0, 0);
    return 0;
}
}  // namespace

int main() {
    for (int k = 16; k <= 320; k += 16)
        for (int stride = k; stride <= k + 64; stride += 16)
            for (int pixels : {1, 2, 31, 32, 33, 34, 65, 225, 289, 961, 1089})
                for (int mt : {1, 2})
                    for (int es : {1, 2, 4}) {
                        if (walk(k, stride, false, pixels, mt, es)) return 1;
                        if (k % 32 == 0 && walk(k, stride, true, pixels, mt, es)) return 1;
                    }
    for (int k : {80, 144, 255, 8})  // strides of eight channels (half values), ragged channel counts
        for (int pixels : {1, 33})
            for (int mt : {1, 2})
                if (walk(k, (k + 7) / 8 * 8, false, pixels, mt, 2)) return 1;
    std::printf("%lld accesses\n", checked);
    return 0;
}
