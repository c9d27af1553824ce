// The output of a 3x3 layer as one list of pixels, which the kernels that stage the input under a run of them share (conv_f32_thirds.hip, conv_staged.hip): the
// vertical strips of all maps, row by row. So ragged maps waste no lanes, small maps of several images share groups, and what a run needs of the input are whole
// rows of a strip, one after another, whatever the run begins with.
#pragma once
#include <algorithm>

#include "common.h"

struct exhip_strips {
    int width = 0, count = 0;  // columns of a strip, strips of a map
    int staged = 0;            // pixels that a run stages at most
    long long tiles = 0;       // runs
};

// The strips for runs of `run` pixels: of all widths that split the map evenly the one whose runs, weighed with what they stage, are least, among those of at most `most`
// staged pixels where there are any. `groups`: of each run, where what counts is the runs that one of 256 CUs gets (0: all of them). `wide`: strips of a column that does
// not exist beside the map's only one.
inline exhip_strips exhip_choose_strips(int out_h, int out_w, int stride, long long images, int run, int most, long long groups, bool wide = false) {
    exhip_strips best;
    double best_cost = 0;
    for (int width = wide ? 2 : out_w;;) {
        const int count = (out_w + width - 1) / width;
        if (!wide) width = (out_w + count - 1) / count;  // the narrowest of that many
        const long long tiles = ((long long)count * width * out_h * images + run - 1) / run;
        // rows that a run touches beside its first, maps that it enters beside its first, and their rows and columns with the border
        const int rows = run % width == 0 ? run / width - 1 : (run + width - 2) / width;
        const int crossed = (int)std::min<long long>((rows + out_h - 1) / out_h, images * count - 1);
        const int staged = (rows * stride + crossed * (3 - stride) + 3) * ((width - 1) * stride + 3);
        const double cost = (staged > most ? 1e18 * staged : 0.) + (double)(groups ? (tiles * groups + 255) / 256 : tiles) * (run + 0.2 * staged);
        if (best.width == 0 || cost < best_cost) {
            best.width = width; best.count = count; best.staged = staged; best.tiles = tiles;
            best_cost = cost;
        }
        if (wide || (width <= 4 && (width == 1 || best.staged <= most))) return best;
        --width;
    }
}

struct exhip_strip_list {
    unsigned total;                // pixels of the list (strips of a ragged width count their missing columns)
    unsigned strip_w, strips;
    exhip_divisor by_strip_w, by_height, by_strips, by_rows, by_cols;
    int staged_rows, staged_cols;  // input rows of a map and columns of a strip with their border

    void set(const exhip_strips& s, int out_h, int stride, long long images) {
        strip_w = (unsigned)s.width; strips = (unsigned)s.count;
        total = (unsigned)((long long)s.width * s.count * out_h * images);
        staged_rows = (out_h - 1) * stride + 3; staged_cols = (s.width - 1) * stride + 3;
        by_strip_w.set(strip_w); by_strips.set(strips); by_height.set((unsigned)out_h);
        by_rows.set((unsigned)staged_rows); by_cols.set((unsigned)staged_cols);
    }

    // The pixel at a place of the list: its number in the output (all ones: none), its first row of all staged ones and its column of the strip.
    struct Where {
        unsigned pix;
        int row, x;
    };
    template <int S>
    __device__ __forceinline__ Where where(unsigned at, int out_h, int out_w) const {
        const unsigned in = at < total ? at : total - 1, row = by_strip_w(in), map = by_height(row), img = by_strips(map);
        const unsigned col = in - row * strip_w, y = row - map * (unsigned)out_h, x = (map - img * strips) * strip_w + col;
        Where w;
        w.row = (int)(map * (unsigned)staged_rows + y * S);
        w.x = (int)col;
        w.pix = at < total && x < (unsigned)out_w ? (img * (unsigned)out_h + y) * (unsigned)out_w + x : 0xffffffffu;
        return w;
    }

    // Where the input pixel at place i of the rows staged from first_row on lies, `none` where that is outside the image. At stride 2 a row's even columns come first, so that
    // neighbouring pixels' taps are neighbours.
    template <int S>
    __device__ __forceinline__ unsigned staged_pixel(int i, int first_row, int in_h, int in_w, int pad_t, int pad_l, int pixel_b, unsigned none) const {
        const unsigned r = by_cols((unsigned)i), row = (unsigned)first_row + r, map = by_rows(row), img = by_strips(map);
        int c = i - (int)r * staged_cols;
        if constexpr (S == 2) c = c < (staged_cols + 1) >> 1 ? 2 * c : 2 * (c - ((staged_cols + 1) >> 1)) + 1;
        const int y = (int)(row - map * (unsigned)staged_rows) - pad_t, x = (int)((map - img * strips) * strip_w) * S + c - pad_l;
        const bool in = (unsigned)y < (unsigned)in_h && (unsigned)x < (unsigned)in_w;
        return in ? ((img * (unsigned)in_h + (unsigned)y) * (unsigned)in_w + (unsigned)x) * (unsigned)pixel_b : none;
    }
};
