// The block width of the streamed decode cells (iu8_stream.h): the host's launch law lays the grid out by it, and the kernels
// follow the grid; and where a launch that shares K counts. Plain C++: the host includes it as it is.
#pragma once

// A symbol of eight k-waves carries two cells: its own (NT 16-column tiles a block, D steps in flight), and 64-column blocks
// of one step in flight, taken for a launch that shares K over workgroups and where they halve the blocks a CU: a block's rows
// cost a CU as much as its weights (iu8_stream.h), and twice the columns share them. us, own cell / 64-column blocks, W4: 32 rows
// of 16384 x 5120 / 2048 / 1024 12.3 / 6.8 / 6.2 -> 10.2 / 6.1 / 4.8, 12288 x 5120 12.6 -> 11.2, 8208 x 5120 10.8 -> 9.9; W8 12288 x 5120
// 17.1 -> 15.1, 16384 x 5120 17.4 -> 16.7. On three shares of K: 5120 x 17408 at 16 / 32 rows 12.8 / 14.5 -> 11.2 / 12.7.
//
// (Symbols whose own blocks are 16 columns wide, more than 32 rows: from 8,192 columns on, where they are more than two a CU.)
// A 64-column block takes 1.75 times one of 32. The busiest CU of 256 runs ceil(n / 8,192) of those: an even count is half as
// many wide ones, an odd one rounds up and loses. W4 at 5 / 16 rows: 17408 x 8192 15.9 / 18.2 -> 19.1 / 20.2, 17408 x 17408 30.2
// -> 36.1, 34816 x 8192 24.9 -> 29.3, W8 18064 x 10112 33.2 -> 38.6 (three and five blocks a CU: own); 9600 x 8192 11.4 -> 9.9, W8 19.7
// -> 16.0, 27648 x 5376 14.9 / 17.1 -> 14.4 / 15.4, W8 27648 x 12288 57.3 -> 52.9 (two and four: wide). Towards the last columns of an even
// count the launch is bound by its bytes and up to eight rows have nothing left to share: 32752 x 12288 at 5 rows 0.97; in front of
// them, past four blocks a CU, 24592 x 6144 0.95. A K of whole 8,192 puts a block's tiles 64 KiB apart and four of them on one channel:
// 16384 / 28672 / 32752 x 8192 at 5 rows 0.93 / 0.97 / 0.90, at 16 rows 1.03 / 1.09 / 1.00, W8 0.97 / 1.04 / 0.97
// (at 24 rows 16384 x 8192 15.6 -> 13.9).
constexpr int IU8_STREAM_WIDE_NT = 4;
constexpr long IU8_STREAM_ROUND = 8192;                                    // columns of one 32-column block a CU
constexpr long IU8_STREAM_FEW_ROWS = 8, IU8_STREAM_FEW_LAST[2] = {8704, 13312};  // `last` in (8704, 13312] at up to eight rows
constexpr long IU8_STREAM_ALIGNED_K = 8192, IU8_STREAM_ALIGNED_ROWS = 16, IU8_STREAM_ALIGNED_LAST = 15360;
constexpr bool iu8_stream_wide(int kw, int own, long m, long n, long k, long ks) {
  if (kw != 8 || ks > 1) return kw == 8;
  if (own < 32) return n > IU8_STREAM_ROUND;
  // own blocks on the busiest CU; columns of its last two
  const long a_cu = (n + IU8_STREAM_ROUND - 1) / IU8_STREAM_ROUND, last = n - (a_cu - 2) * IU8_STREAM_ROUND;
  const bool aligned = k % IU8_STREAM_ALIGNED_K == 0;
  if (a_cu % 2) return false;
  if (m > IU8_STREAM_FEW_ROWS) return m > IU8_STREAM_ALIGNED_ROWS || !aligned || last <= IU8_STREAM_ALIGNED_LAST;
  if (a_cu == 2) return !aligned || last <= IU8_STREAM_FEW_LAST[1];
  return !aligned && last > IU8_STREAM_FEW_LAST[0] && last <= IU8_STREAM_FEW_LAST[1];
}

// Where a block of a launch that shares K counts its arrivals: in a word of its own, or, where `two`, two blocks in one word, 16 bits
// each, so that a 64-column launch's counters fit where a 128-column tile launch's would (rules.cpp:stream_in_tile_workspaces). A word
// a block is the faster one, 2-5 % of a launch (us, two / one: 9 rows of 3184 x 10368 7.89 / 7.50, 16 of 5120 x 10240 8.73 / 8.38, 36 10.84 / 10.57,
// 48 of 5120 x 12288 11.97 / 11.75; int8 and K = 17,408 1-2 % or level), so words are shared only by the launches that may stand in such workspaces; and never where
// the shares pass 16 bits (a K of 8.4 million and more, which a pair's halves and a symbol by name take).
constexpr bool iu8_stream_shared_words(bool w8, int tm, long k) { return !w8 && tm >= 3 && k >= 16384; }
struct iu8_arrival {
  int word;
  unsigned shift, mask;
  constexpr unsigned one() const { return 1u << shift; }
  constexpr bool last(unsigned before, int shares) const { return ((before >> shift) & mask) == (unsigned)(shares - 1); }
  constexpr unsigned all(int shares) const { return (unsigned)shares << shift; }
};
constexpr iu8_arrival iu8_arrival_of(int block, int shares, bool two = true) {
  return two && shares <= 0xFFFF ? iu8_arrival{block >> 1, (block & 1) * 16u, 0xFFFFu} : iu8_arrival{block, 0u, ~0u};
}
