// The block width of the streamed decode cells (iu8_stream.h), one rule for the kernels and for the host's launch law. Plain
// C++: the host includes it as it is.
#pragma once

// A symbol of eight k-waves carries two cells: its own (NT 16-column tiles a block, D steps in flight), and 64-column blocks
// of one step in flight, taken where its own would be more than one round of the 256 CUs (8,192 columns of 32) and for a
// launch that shares K over workgroups: a block's rows cost a CU as much as its weights (iu8_stream.h), and twice the columns
// share them. us, own cell / 64-column blocks, W4: 32 rows of 16384 x 5120 / 2048 / 1024 12.3 / 6.8 / 6.2 -> 10.2 / 6.1 / 4.8, 12288 x
// 5120 12.6 -> 11.2, 8208 x 5120 10.8 -> 9.9; W8 12288 x 5120 17.1 -> 15.1, 16384 x 5120 17.4 -> 16.7. On three shares of K: 5120 x
// 17408 at 16 / 32 rows 12.8 / 14.5 -> 11.2 / 12.7.
constexpr int IU8_STREAM_WIDE_NT = 4;
constexpr bool iu8_stream_wide(int kw, int n, int ks) { return kw == 8 && (ks > 1 || n > 32 * 256); }
