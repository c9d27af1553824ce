// Where the waves of the pointwise kernels (conv_pw.hip) read shortcuts from and store results to: plain arithmetic without a
// GPU type, so that a host program can walk it over shapes.
//
// A wave handles 32 pixels ("rows") x 32-channel blocks of a pixel-major tensor through a buffer view that begins at its first
// row and channel and ends behind its last row. Whatever lies beyond the view reads zeros and is not stored, so a lane with
// nothing to do gets an offset beyond every view -- which takes a view of less than kPwOutOfRange bytes. The size is an
// unsigned word to the hardware: a negative one would be a view of nearly 4 GiB that holds that offset too.
#pragma once

constexpr int kPwOutOfRange = 0x7ffff000;

// Channels from here on are not written. `exact`: the results lie inside a wider tensor, whose other channels are another layer's.
constexpr int pw_channel_end(int k, int k_stride, bool exact) { return exact || k_stride < k ? k : k_stride; }

// Whether a 32-channel block holds a channel that is written: the last group of blocks may reach beyond the last one.
constexpr bool pw_block_exists(int kb, int channel_end) { return kb * 32 < channel_end; }

// Bytes of the view of `rows` rows from channel byte ch_bytes on; empty where that lies behind the last row's end.
constexpr int pw_view_bytes(int rows, int row_bytes, int ch_bytes) { return rows * row_bytes > ch_bytes ? rows * row_bytes - ch_bytes : 0; }

// A lane's offset in the view: `byte` bytes into its row, of the `bytes` that the row has left from the view's channel on.
constexpr int pw_lane_offset(int row, int row_bytes, int byte, int bytes) { return byte < bytes ? row * row_bytes + byte : kPwOutOfRange; }

// The view, the offsets in it and the next 31 rows' stay below kPwOutOfRange.
constexpr bool pw_row_fits(long long row_bytes) { return row_bytes * 64 < kPwOutOfRange; }
