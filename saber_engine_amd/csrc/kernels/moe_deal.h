// How the routed tile launches deal their work items over the workgroups (moe_iu8.gfx950.hip). Plain C++: a test compiles it
// on the host.
#pragma once

// hi heavy items, li light ones, G positions. Heavy item w + r * G is position w's, so the first `more` positions have one more
// of them than the rest, and take `cost` light items less for it (a heavy item stands for `cost` light ones). Rounds of light
// items below l_more go to all positions, the ones from there to l_rest to the rest, each dealt from the last position down.
// Dealt evenly, the two kinds apart, a position with the odd heavy item had a full share of light ones behind it, and the launch
// waited for those: a shared expert's 24 heavy items at 300 tokens, a layer of 291 us -> 282, at 500 / 700 tokens 313 / 334 ->
// 300 / 316 (cost 1: 289 / 313 / 332, cost 3: 282 / 301 / 316; one position in ten of a launch at 1,000 tokens: 2 against 3 329 / 334).
// A 256-row item stands for 4 (2: 820 us at 4,000 tokens with a shared expert, 3: 823, 4 and 5: 816; without one level).
struct moe_deal {
  int more, l_more, l_rest;
  constexpr int light_id(int r, int w, int G) const {
    return (r < l_more ? r : l_more) * G + (r > l_more ? r - l_more : 0) * (G - more) + G - 1 - w;
  }
};
constexpr moe_deal moe_deal_of(int hi, int li, int G, int cost) {
  const int more = hi % G, rest = G - more;
  const int l = li <= rest * cost ? (li + rest - 1) / rest : (li + more * cost + G - 1) / G;
  return moe_deal{more, l > cost ? l - cost : 0, l};
}
// How many of nt tiles, `heavy` of them heavy, run on the tile cell in a kernel that does not pass over its item table again and
// again: all of them, the light ones behind the heavy ones, where the light items are more a position than the table holds.
constexpr int moe_tile_cell_tiles(int heavy, int nt, int gx, int G, int cost, int light_rounds) {
  return moe_deal_of(heavy * gx, (nt - heavy) * gx, G, cost).l_rest > light_rounds ? nt : heavy;
}
