// How a launch of the 256 x 256 tile cell lays its rows out, one rule for the kernel and for the host's estimate of it. Plain C++:
// the host includes it as it is.
#pragma once

// G workgroups, gx column blocks, m rows; times in hundredths of a 256 x 256 tile's.
//   tail  the last round's tiles as quarter tiles on the 128 x 128 cell, where they are at most half the workgroups: 42 a
//         round of quarter tiles
//   thin  the rows past the last whole 256, at most 128 of them, on 128 x 256 tiles of their own (`gx` of them; int4 weights:
//         30 for up to 32 rows, whose waves run one row block of four, else 58) behind the whole tiles, first on the workgroups with a tile
//         less -- in place of whole tiles, which multiply the padding as well: 777 rows of 34816 x 5120 are 408 tiles and 136
//         thin ones instead of 544. Taken where the count says that it is shorter, behind quarter tiles by more than 15 (a third
//         phase: 1,540 rows of 12288 x 2048, 172 for 184, 49.9 -> 52.0 us), from K = 1,024 (below, a tile is fill and epilogue:
//         1,050 rows of 34816 x 256 23.5 -> 25.3 us). us, whole tiles / thin, 34816 x 5120: 520 / 777 / 1,030 / 1,300 / 1,800 /
//         4,120 / 8,200 rows 123.9 / 150.1 / 189.1 / 215.8 / 282.0 / 604.7 / 1,162 -> 109.6 / 134.8 / 173.5 / 198.0 / 262.3 / 578.9 /
//         1,136; against the cell that the law had there: 264 rows 81.0 -> 71.7, 520 of 24576 x 4096
//         69.1 -> 58.8, 1,030 of 14336 x 5120 82.3 -> 71.7, 3,100 of 5120 x 5120 / 6144 / 17408 78.1 / 90.7 / 237.0 -> 71.3 / 83.2 /
//         215.3; level (0-3 %) where the rows past 256 are 65-128 and the count is close.
//         Int8 weights are twice the bytes under the same few rows: a thin tile takes 65 and 80, and none of it hides behind a whole
//         tile. They are taken behind whole rounds, or where the workgroups with a tile less hold all of them, whole tiles / thin:
//         4,105 / 4,200 rows of 20480 x 5120 386 / 387 -> 368 / 368, 8,212 of 28672 x 5120 1,046 -> 1,016, 777 / 800 of 34816 x 5120 153.2 /
//         153.7 -> 149.7 / 149.3, 1,030 of 28672 x 5120 155.9 -> 148.6, 3,100 of 10240 x 5120 149.3 -> 138.6; laid out by int4's figures they
//         lost: 520 rows of 28672 x 5120 108 -> 124, 1,030 of 16384 x 5120 94 -> 104, 4,105 of 8192 x 5120 152 -> 164 (234 launches of
//         thirteen widths x five K, weights from memory: none slower than its whole tiles by more than the runs differ).
struct iu8_pf_plan {
  bool tail, thin;
  int gy;                // row blocks of whole tiles
  int q, rem;            // whole tiles: q rounds and rem tiles
  int own, own_wgs;      // thin tiles: the first own * own_wgs go to the own_wgs workgroups behind `rem`, `own` each
  int cost;
};

constexpr int iu8_ceil_div(int a, int b) { return (a + b - 1) / b; }
constexpr iu8_pf_plan iu8_pf_plan256(int m, int gx, int G, int k, bool w8) {
  constexpr int QUARTER = 42;
  iu8_pf_plan p{};
  p.gy = iu8_ceil_div(m, 256);
  p.q = gx * p.gy / G, p.rem = gx * p.gy % G;
  p.tail = p.q >= 1 && p.rem > 0 && 2 * p.rem <= G;
  p.cost = 100 * p.q + (p.tail ? QUARTER * iu8_ceil_div(4 * p.rem, G) : p.rem ? 100 : 0);
  const int live = m % 256, full = m / 256;
  if (live == 0 || live > 128 || full == 0 || k < 1024) return p;
  const int x = w8 ? (live <= 32 ? 65 : 80) : live <= 32 ? 30 : 58;
  iu8_pf_plan t{};
  t.thin = true, t.gy = full, t.q = gx * full / G, t.rem = gx * full % G;
  t.own_wgs = t.rem ? G - t.rem : 0;
  if (w8) {  // every thin tile on a workgroup with a tile less, or on all of them behind whole rounds
    t.own = t.rem ? iu8_ceil_div(gx, t.own_wgs) : 0;
    const int own = t.own * x;
    t.cost = 100 * t.q + (!t.rem ? x * iu8_ceil_div(gx, G) : own > 100 ? own : 100);
    return t.cost < p.cost ? t : p;
  }
  if (t.q >= 1 && t.rem > 0 && 2 * t.rem <= G) {
    iu8_pf_plan u = t;
    u.own_wgs = 0;
    u.tail = true, u.cost = 100 * t.q + QUARTER * iu8_ceil_div(4 * t.rem, G) + x * iu8_ceil_div(gx, G);
    if (u.cost + 15 < p.cost) p = u;
  }
  t.own = t.rem ? 100 / x : 0;
  const int left = gx - t.own * t.own_wgs;
  t.cost = 100 * (t.q + (t.rem > 0)) + (left > 0 ? x * iu8_ceil_div(left, G) : 0);
  return t.cost < p.cost ? t : p;
}
